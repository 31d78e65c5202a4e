"""Patches of whole SOR sweeps (ufemism_amd/csrc/patch_host.h) on the CPU.

The builder is compiled with g++ and driven on generated meshes.  Sweeping
every patch on its own (own rows and recomputed halo rows, in the list's local
indices, as the device kernel does) must give every point the bits of sweeps
over the whole mesh: the same operations on the same values.  The packed
indices, the group bounds that the kernel relies on and the list's layout are
checked on the way.
"""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from oracle import pyoracle as po
from ufemism_amd import geometry, meshgen

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ufemism_amd", "csrc")

DRIVER = r"""
#include "patch_host.h"
#include <cstring>
using namespace ufe;
// one relaxation of a row: an order-dependent chain of products and a quotient
static double relax(const PatchMesh &m, int p, const double *coef, const double *rhs, double own, const double *x, int n) {
  double s = 0.0;
  const int64_t b = m.cptr[p >> 6] + (p & 63);
  for (int k = 0; k < n; k++) s = s + coef[b + 64 * (int64_t)k] * x[k];
  return own - 1.3 * ((s - rhs[p] + 2.0 * own) / 2.0);
}
extern "C" long check(int nA, const int *cs, const int *ca, const int64_t *cptr, const uint8_t *deg, const int32_t *col,
                      int n_neu, const int32_t *nr, const int32_t *np_, const int32_t *nc, int n_cor, const int32_t *kr,
                      const int32_t *kp, const int32_t *kc, const uint32_t *key, const uint16_t *member, int own, int nu,
                      int backward, int neumann, int ring, const double *coef, const double *rhs, const double *x0,
                      double *stats) {
  const PatchMesh m{nA, cs, ca, cptr, deg, col, n_neu, n_cor, nr, np_, nc, kr, kp, kc, key, member};
  const std::vector<int32_t> order = patch_order(m);
  std::vector<char> seen(nA, 0);
  for (int32_t p : order) seen[p]++;
  for (int p = 0; p < nA; p++)
    if (seen[p] != 1) return -1;
  // the whole mesh
  std::vector<double> X(x0, x0 + nA), xs(32);
  for (int s = 0; s < nu; s++)
    for (int j = 0; j < 5; j++) {
      const int c = backward ? 4 - j : j;
      for (int p = cs[c]; p < cs[c] + ca[c]; p++) {
        const int64_t b = cptr[p >> 6] + (p & 63);
        for (int k = 0; k < deg[p]; k++) xs[k] = X[col[b + 64 * (int64_t)k]];
        X[p] = relax(m, p, coef, rhs, X[p], xs.data(), deg[p]);
      }
    }
  if (neumann)
    for (int w = 0; w < 2; w++) {
      const int n = w ? n_cor : n_neu;
      const int32_t *row = w ? kr : nr, *ptr = w ? kp : np_, *cl = w ? kc : nc;
      for (int i = 0; i < n; i++) {
        double t = 0.0;
        for (int a = ptr[i]; a < ptr[i + 1]; a++) t = t + X[cl[a]];
        X[row[i]] = t / (double)(ptr[i + 1] - ptr[i]);
      }
    }
  std::vector<double> Y(nA, 0.0);
  std::vector<char> sor(nA, 0);
  for (int c = 0; c < 5; c++)
    for (int p = cs[c]; p < cs[c] + ca[c]; p++) {
      sor[p] = 1;
      const int64_t b = cptr[p >> 6] + (p & 63);
      for (int k = 0; k < deg[p]; k++) Y[p] += coef[b + 64 * (int64_t)k] * X[col[b + 64 * (int64_t)k]];
    }
  std::vector<PatchHost> parts;
  if (!patch_build(m, order, own, nu, backward != 0, neumann != 0, ring != 0, parts)) return -2;
  // the points that patches exchange between sweeps, marked in a copy
  {
    std::vector<PatchHost> shared = parts;
    patch_mark_shared(nA, shared);
    std::vector<char> read(nA, 0), marked(nA, 0);
    size_t list0 = 0;
    for (size_t q = 0; q < parts.size(); q++) {
      for (const PatchDesc &d : parts[q].d)
        for (int i = 0; i < d.nlist; i++) {
          const int32_t p = parts[q].rows[d.list - list0 + i], s = shared[q].rows[d.list - list0 + i];
          if ((s & 0x7fffffff) != p) return -11;
          if (i >= d.ncs + d.ne + d.nk) read[p] = 1;
          if (s < 0) marked[p]++;
        }
      list0 += parts[q].rows.size();
    }
    for (int p = 0; p < nA; p++)
      if (read[p] != marked[p]) return -12;
  }
  PatchHost H;
  auto join = [](auto &a, auto &b) { a.insert(a.end(), b.begin(), b.end()); };
  for (PatchHost &q : parts) {
    join(H.d, q.d);
    join(H.rows, q.rows);
    join(H.nptr, q.nptr);
    join(H.sbase, q.sbase);
    join(H.lcol, q.lcol);
    join(H.ov_e, q.ov_e);
    join(H.ovf, q.ovf);
    join(H.ov_c, q.ov_c);
    join(H.ncol, q.ncol);
    H.max_list = std::max(H.max_list, q.max_list);
    H.max_group = std::max(H.max_group, q.max_group);
    H.max_ov = std::max(H.max_ov, q.max_ov);
  }
  std::vector<int> wrote(nA, 0);
  long bad = 0;
  double computed = 0.0, listed = 0.0;
  for (const PatchDesc &d : H.d) {
    if (d.list < 0 || d.list + (size_t)d.nlist > H.rows.size() || d.comp + (size_t)d.ncs > H.sbase.size() ||
        3 * ((size_t)d.comp + d.ncs) > H.lcol.size() || d.ov + (size_t)d.nov > H.ov_e.size() ||
        d.nlist > H.max_list || d.nov > H.max_ov || d.ncs + d.ne + d.nk > d.nlist)
      return -3;
    if (neumann && d.nptr + (size_t)d.ne + d.nk + 1 > H.nptr.size()) return -4;
    computed += d.ncs;
    listed += d.nlist;
    std::vector<double> v(d.nlist);
    for (int i = 0; i < d.nlist; i++) v[i] = x0[H.rows[d.list + i]];
    auto gather = [&](int l, double *x) {
      const uint32_t sb = H.sbase[d.comp + l];
      const int n = sb >> PATCH_BASE_BITS, p = H.rows[d.list + l];
      if (n != deg[p] || (int64_t)(sb & ((1u << PATCH_BASE_BITS) - 1)) != cptr[p >> 6] + (p & 63)) return -1;
      for (int s = 0; s < n; s++) {
        int q;
        if (s < 6) q = (H.lcol[3 * (size_t)d.comp + (size_t)(s / 2) * d.ncs + l] >> (16 * (s & 1))) & 0xffff;
        else {
          const int o = d.ov + H.ovf[d.comp + l] + s - 6;
          if (o >= d.ov + d.nov || H.ov_e[o] != (sb & ((1u << PATCH_BASE_BITS) - 1)) + 64u * s) return -1;
          q = H.ov_c[o];
        }
        if (q >= d.nlist || H.rows[d.list + q] != col[cptr[p >> 6] + (p & 63) + 64 * (int64_t)s]) return -1;
        x[s] = v[q];
      }
      return n;
    };
    for (int s = 0; s < nu; s++)
      for (int j = 0; j < 5; j++) {
        const int c = backward ? 4 - j : j;
        if (d.own[c] > d.cnt[c][nu - 1] || d.cnt[c][0] > H.max_group || (nu == 2 && d.cnt[c][1] > d.cnt[c][0]) ||
            d.g[c] + d.cnt[c][0] > d.ncs)
          return -5;
        for (int t = 0; t < d.cnt[c][s]; t++) {
          const int l = d.g[c] + t, n = gather(l, xs.data());
          if (n < 0) return -6;
          v[l] = relax(m, H.rows[d.list + l], coef, rhs, v[l], xs.data(), n);
        }
      }
    if (neumann)
      for (int e = 0; e < d.ne + d.nk; e++) {
        double t = 0.0;
        const int a0 = H.nptr[d.nptr + e], a1 = H.nptr[d.nptr + e + 1];
        if (a0 < 0 || a1 <= a0 || (size_t)a1 > H.ncol.size()) return -7;
        for (int a = a0; a < a1; a++) {
          if (H.ncol[a] >= d.nlist) return -8;
          t = t + v[H.ncol[a]];
        }
        v[d.ncs + e] = t / (double)(a1 - a0);
      }
    auto own_out = [&](int l) {
      const int p = H.rows[d.list + l];
      wrote[p]++;
      if (std::memcmp(&v[l], &X[p], 8)) bad++;
      if (ring && sor[p]) {
        const int n = gather(l, xs.data());
        double y = 0.0;
        const int64_t b = cptr[p >> 6] + (p & 63);
        for (int k = 0; k < n; k++) y += coef[b + 64 * (int64_t)k] * xs[k];
        if (std::memcmp(&y, &Y[p], 8)) bad++;
      }
    };
    for (int c = 0; c < 5; c++)
      for (int t = 0; t < d.own[c]; t++) {
        if (t && H.rows[d.list + d.g[c] + t] != H.rows[d.list + d.g[c] + t - 1] + 1) return -9;   // contiguous
        own_out(d.g[c] + t);
      }
    for (int e = 0; e < d.ne + d.nk; e++)
      if (e < d.own_e || (e >= d.ne && e < d.ne + d.own_k)) own_out(d.ncs + e);
  }
  for (int p = 0; p < nA; p++)
    if (wrote[p] != 1) return -10;
  stats[0] = computed / nA;
  stats[1] = listed / nA;
  return bad;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("patch")
    (d / "check.cpp").write_text(DRIVER)
    so = d / "check.so"
    subprocess.run([cxx, "-std=c++17", "-O2", "-ffp-contract=off", "-Wall", "-Wextra", "-Wno-unused-parameter", "-fPIC", "-shared", "-pthread", f"-I{CSRC}",
                    str(d / "check.cpp"), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


def colour_order(mesh, members=1):
    """The colour-ordered points of `members` copies of a mesh, as ufe_mesh_upload lays them out."""
    om = po.OracleMesh(mesh).build()
    n1 = om.nVAaAc
    nc, C, colour = (np.tile(om[k], (members,) + (1,) * (om[k].ndim - 1)) for k in ("nCAaAc", "CAaAc", "colour"))
    off = np.repeat(np.arange(members) * n1, n1)
    edge = np.tile(np.concatenate([mesh.edge_index, om["edge_index_Ac"]]) > 0, members)
    corner = np.tile(np.arange(n1) < 4, members)
    V = np.tile(om["VAaAc"], (members, 1))
    lo, span = V.min(0), (V.max(0) - V.min(0)).max()
    g = ((V - lo) / span * 65535).astype(np.int64)
    key = meshgen._hilbert_index(g[:, 0], g[:, 1]).astype(np.uint32)
    member = (off // n1).astype(np.uint16)
    n = len(nc)
    perm, start, active = [], [], []
    for c in range(1, 6):
        rows = np.nonzero((colour == c) & ~edge)[0]
        rest = np.nonzero((colour == c) & edge)[0]
        start.append(sum(map(len, perm)))
        active.append(len(rows))
        perm += [rows[np.lexsort((rows, key[rows], member[rows]))], rest]
    perm = np.concatenate(perm)
    iperm = np.empty(n, np.int64)
    iperm[perm] = np.arange(n)
    nchunk = (n + 63) // 64
    deg = nc[perm].astype(np.uint8)
    width = np.array([deg[64 * k:64 * k + 64].max() for k in range(nchunk)], np.int64)
    cptr = np.concatenate([[0], np.cumsum(width * 64)]).astype(np.int64)
    base = cptr[np.arange(n) // 64] + np.arange(n) % 64
    col = np.zeros(cptr[-1], np.int32)
    neigh = lambda a: C[a, :nc[a]] - 1 + off[a]  # noqa: E731
    for s in range(int(deg.max())):
        rows = np.nonzero(deg > s)[0]
        a = perm[rows]
        col[base[rows] + 64 * s] = iperm[C[a, s] - 1 + off[a]]

    def lists(points, keep):
        row, ptr, cl = [], [0], []
        for a in points:
            cl += [iperm[j] for j in neigh(a) if keep(j)]
            row.append(iperm[a])
            ptr.append(len(cl))
        return [np.array(x, np.int32) for x in (row, ptr, cl)]

    neu = lists(np.nonzero(edge & ~corner)[0], lambda j: not edge[j])
    cor = lists(np.nonzero(corner)[0], lambda j: True)
    return dict(n=n, start=np.array(start + [n], np.int32), active=np.array(active, np.int32), cptr=cptr, deg=deg, col=col,
                neu=neu, cor=cor, key=key[perm].copy(), member=member[perm].copy() if members > 1 else None)


MESHES = {"dummy": lambda: colour_order(meshgen.dummy_mesh()),
          "dome600": lambda: colour_order(geometry.dome(600, seed=3).mesh),
          "marine5k": lambda: colour_order(geometry.marine(5000, seed=8).mesh),
          "two_members": lambda: colour_order(geometry.marine(1500, seed=4).mesh, members=2),
          "marine20k": lambda: colour_order(geometry.marine(20000, seed=5).mesh)}   # over 65,536 points: several threads
_cache = {}


@pytest.mark.parametrize("name", sorted(MESHES))
@pytest.mark.parametrize("own,nu,backward,neumann,ring", [
    (1, 1, 0, 1, 0), (31, 1, 0, 1, 0), (124, 1, 0, 1, 0), (500, 2, 0, 1, 1), (500, 2, 1, 1, 1), (77, 2, 1, 1, 1),
    (128, 1, 1, 1, 1), (200, 2, 0, 0, 0), (200, 2, 1, 0, 0), (100000, 2, 0, 1, 1)])
def test_patch_sweeps_equal_whole_sweeps(lib, name, own, nu, backward, neumann, ring):
    m = _cache.setdefault(name, None) or _cache.setdefault(name + "!", MESHES[name]())
    _cache[name] = m
    if m["n"] > 20000 and (own == 1 or own > 60000):
        pytest.skip("sizes of the small meshes")
    rng = np.random.default_rng(own + nu)
    coef, rhs, x0 = rng.standard_normal(len(m["col"])), rng.standard_normal(m["n"]), rng.standard_normal(m["n"])
    ptr = lambda a: None if a is None else ctypes.c_void_p(np.ascontiguousarray(a).ctypes.data)  # noqa: E731
    stats = (ctypes.c_double * 2)()
    own = min(own, m["n"])
    lib.check.restype = ctypes.c_long
    bad = lib.check(m["n"], ptr(m["start"]), ptr(m["active"]), ptr(m["cptr"]), ptr(m["deg"]), ptr(m["col"]),
                    len(m["neu"][0]), *map(ptr, m["neu"]), len(m["cor"][0]), *map(ptr, m["cor"]), ptr(m["key"]),
                    ptr(m["member"]), own, nu, backward, neumann, ring, ptr(coef), ptr(rhs), ptr(x0), stats)
    print(f"  {name} own {own}: {stats[0]:.2f} rows computed and {stats[1]:.2f} points listed per own point", flush=True)
    assert bad == 0, bad
