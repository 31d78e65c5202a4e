// Patches of the colour-ordered AaAc points: contiguous pieces of the Hilbert
// order, each with the halo rows that a whole SOR sweep of its own rows
// depends on.  A kernel that holds one patch per workgroup then runs every
// colour of a sweep (and the Neumann update after it) without waiting for
// another workgroup: a halo row is recomputed by each patch that needs it, from
// the same values with the same operations.
//
// The halo of a sweep is small because a colour pass only reads rows of earlier
// colours that this sweep has already updated: walking back from the own rows,
// each step leads to an earlier colour.  On the generator's meshes a patch of
// 1,024 points computes 1.17 rows per own row for one sweep and 1.6 for two,
// and reads 1.4 or 1.9 points (124 points: 1.5 and 2.9).
//
// Plain C++ (no HIP types) so that the CPU tests compile it on their own.
#pragma once

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <new>
#include <vector>

#include "amg_host.h"

namespace ufe {

// One patch.  Its point list is [rows of colour 1 .. 5][edge points][corners]
// [points only read]; a position in that list is a local index.  Inside a
// colour the own rows come first, then the halo rows by how many of the sweeps
// compute them.
struct PatchDesc {
  int32_t list, nlist;            // rows[list .. list + nlist): colour-order indices of the points
  int32_t comp, ncs;              // SOR rows computed: sbase / ovf [comp ..], lcol [3 comp ..] (three planes of ncs)
  int32_t ov, nov;                // slots beyond the sixth
  int32_t nptr;                   // first of the ne + nk + 1 offsets into ncol
  int32_t ne, nk, own_e, own_k;   // edge points and corners, own ones first
  int32_t g[5], own[5];           // first local index and own rows of a colour
  int32_t cnt[5][2];              // rows of a colour computed in the first and in the second sweep
};

struct PatchMesh {                // the colour-ordered points (see ufe_mesh_upload)
  int nA;
  const int *colour_start, *colour_active;
  const int64_t *cptr;            // SELL-64 neighbour lists
  const uint8_t *deg;
  const int32_t *col;
  int n_neu, n_cor;               // edge points and corners with the points they average
  const int32_t *neu_row, *neu_ptr, *neu_col, *cor_row, *cor_ptr, *cor_col;
  const uint32_t *key;            // Hilbert key of each point
  const uint16_t *member;         // batch member of each point, or null
};

struct PatchHost {                // a part of the patches, one after another
  std::vector<PatchDesc> d;
  std::vector<int32_t> rows, nptr;
  std::vector<uint32_t> sbase, lcol, ov_e;   // sbase: SELL position of the first slot, degree in the top 5 bits
  std::vector<uint16_t> ovf, ov_c, ncol;
  int max_list = 0, max_group = 0, max_ov = 0, max_ncs = 0, max_neu = 0, max_ncol = 0;
};

constexpr int PATCH_BASE_BITS = 27;

// Host threads for the patches of n points: one per 2,048 points (about a third of
// a millisecond of walking), at most the hardware's and 16.  A mesh's first solve
// waits for its patches, and on small meshes a solve takes no longer than a walk on
// one thread.  First solve of a 16k-vertex mesh with the SOR loop / by multigrid
// (the sets side by side beside the multigrid set-up): one thread 7.3 / 38.0 ms, 16
// 3.6 / 21.1, where the colour launches take 4.0 / 25.0.
inline int patch_threads(int64_t n) {
  const unsigned h = std::thread::hardware_concurrency();
  return (int)std::max<int64_t>(1, std::min<int64_t>(n / 2048, std::min(h, 16u)));
}

// The buffers beside the patches: makes those that are not there yet, each on its
// own, so that a call after one that stopped half-way makes the rest.  make(p)
// returns 0, with p still null where there is no room, or an error, which ends
// this; the patches may be used only once every buffer is there.
template <typename Make, typename... P>
inline int patch_spaces(Make make, P *&...p) {
  int r = 0;
  ((r = r || p ? r : make(p)), ...);
  return r;
}

// The least that the largest colour of a patch can hold when np patches share the
// points: a mesh for which this exceeds the workgroup needs no walk to be refused.
inline int patch_least_group(const int *colour_active, int np) {
  int most = 0;
  for (int c = 0; c < 5; c++) most = std::max(most, colour_active[c]);
  return (most + np - 1) / np;
}

// All points along the Hilbert order (member by member): the rows of a colour
// are sorted already, so this is a merge of the five colours and the rest, in
// as many key ranges as there are host threads.
inline std::vector<int32_t> patch_order(const PatchMesh &m) {
  std::vector<int32_t> out(m.nA), rest;
  for (int c = 0; c < 5; c++) {
    const int next = c < 4 ? m.colour_start[c + 1] : m.nA;
    for (int p = m.colour_start[c] + m.colour_active[c]; p < next; p++) rest.push_back(p);
  }
  auto k = [&](int32_t p) { return ((uint64_t)(m.member ? m.member[p] : 0) << 32) | m.key[p]; };
  std::sort(rest.begin(), rest.end(), [&](int32_t a, int32_t b) { return k(a) < k(b) || (k(a) == k(b) && a < b); });
  // first entry of run r (a colour, or 5: the rest) with a key of at least v
  auto at = [&](int r, int i) { return r < 5 ? (int32_t)(m.colour_start[r] + i) : rest[i]; };
  auto len = [&](int r) { return r < 5 ? m.colour_active[r] : (int)rest.size(); };
  auto lower = [&](int r, uint64_t v) {
    int lo = 0, hi = len(r);
    while (lo < hi) {
      const int mid = (lo + hi) / 2;
      if (k(at(r, mid)) < v) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  int big = 0;
  for (int r = 1; r < 6; r++)
    if (len(r) > len(big)) big = r;
  const int parts = patch_threads(m.nA);
  amg_parts(parts, parts, [&](int, int t0, int t1) {
    for (int t = t0; t < t1; t++) {
      int h[6], e[6];
      int64_t o = 0;
      uint64_t hk[6];
      for (int r = 0; r < 6; r++) {
        h[r] = t == 0 ? 0 : lower(r, k(at(big, (int)((int64_t)len(big) * t / parts))));
        e[r] = t + 1 == parts ? len(r) : lower(r, k(at(big, (int)((int64_t)len(big) * (t + 1) / parts))));
        o += h[r];
        hk[r] = h[r] < e[r] ? k(at(r, h[r])) : UINT64_MAX;
      }
      while (true) {
        int b = 0;
        for (int r = 1; r < 6; r++)
          if (hk[r] < hk[b]) b = r;
        if (hk[b] == UINT64_MAX) break;
        out[o++] = at(b, h[b]++);
        hk[b] = h[b] < e[b] ? k(at(b, h[b])) : UINT64_MAX;
      }
    }
  });
  return out;
}

// Patches of own_size points for nu (1 or 2) sweeps in forward or backward
// colour order.  neumann: the edge points and corners are updated after the
// sweeps; ring: the own rows' neighbours are final as well (for A z of the own
// rows).  Built in contiguous parts on the host's threads; the offsets in the
// descriptors count from the start of the first part, so that the parts are
// simply put one after another.  Returns false when the mesh does not fit the
// packed indices, at the first patch with more than group_max rows of a colour, or
// where host memory runs out on one of the threads (an exception must not leave a
// thread).  threads: at most so many (0: patch_threads); the patches do not depend
// on it.
inline bool patch_build(const PatchMesh &m, const std::vector<int32_t> &order, int own_size, int nu, bool backward,
                        bool neumann, bool ring, std::vector<PatchHost> &part, int group_max = INT32_MAX,
                        int threads = 0) {
  const int nA = m.nA, np = (nA + own_size - 1) / own_size;
  part.clear();
  if (m.cptr[(nA + 63) / 64] >= (int64_t)1 << PATCH_BASE_BITS || nu < 1 || nu > 2) return false;
  // kind of a point: colour 0..4 of a SOR row, 5 edge point, 6 corner; place: its entry in the edge or corner list
  std::vector<uint8_t> kind(nA, 5);
  std::vector<std::pair<int32_t, int32_t>> place;
  for (int c = 0; c < 5; c++)
    std::fill(kind.begin() + m.colour_start[c], kind.begin() + m.colour_start[c] + m.colour_active[c], (uint8_t)c);
  for (int i = 0; i < m.n_neu; i++) place.push_back({m.neu_row[i], i});
  for (int i = 0; i < m.n_cor; i++) {
    place.push_back({m.cor_row[i], i});
    kind[m.cor_row[i]] = 6;
  }
  std::sort(place.begin(), place.end());
  auto place_of = [&](int32_t p) {
    const auto it = std::lower_bound(place.begin(), place.end(), std::make_pair(p, (int32_t)-1));
    return it != place.end() && it->first == p ? it->second : -1;
  };
  const int parts = std::min(np, threads > 0 ? threads : patch_threads(nA));
  part.resize(parts);
  std::vector<uint8_t> bad(parts, 0);
  auto walk = [&](int t, int b0, int b1, uint64_t *where) {
    PatchHost &H = part[t];
    const size_t guess = (size_t)(b1 - b0) * own_size * 2;
    H.rows.reserve(guess + guess / 4);
    H.sbase.reserve(guess);
    H.ovf.reserve(guess);
    H.lcol.reserve(3 * guess);
    std::vector<int32_t> pts, pend[7], now, loc, ent;   // ent: the entries of a computed row's neighbours
    std::vector<int64_t> ent0;                          // per entry, -1: not computed
    std::vector<int8_t> sweeps;   // sweeps that compute an entry (0: only read; edge points and corners: 1)
    std::vector<uint8_t> group;
    for (int b = b0; b < b1 && !bad[t]; b++) {
      const uint64_t tag = (uint64_t)(b + 1) << 32;
      pts.clear();
      sweeps.clear();
      ent.clear();
      ent0.clear();
      for (auto &v : pend) v.clear();
      auto enter = [&](int32_t p) -> int32_t {
        const uint64_t w = where[p];
        if ((w >> 32) == (uint64_t)(b + 1)) return (int32_t)(uint32_t)w;
        const int32_t e = (int32_t)pts.size();
        where[p] = tag | (uint32_t)e;
        pts.push_back(p);
        sweeps.push_back(0);
        ent0.push_back(-1);
        pend[kind[p]].push_back(e);
        return e;
      };
      const int q0 = (int)((int64_t)nA * b / np), q1 = (int)((int64_t)nA * (b + 1) / np), nown = q1 - q0;
      for (int q = q0; q < q1; q++) enter(order[q]);
      if (ring)
        for (int i = 0; i < nown; i++)
          if (kind[pts[i]] < 5) {
            const int32_t p = pts[i];
            const int64_t base = m.cptr[p >> 6] + (p & 63);
            for (int s = 0; s < m.deg[p]; s++) enter(m.col[base + (int64_t)s * 64]);
          }
      // back in time: corners, edge points, then the colours of the last sweep, ...
      if (neumann)
        for (int kd : {6, 5})
          for (size_t i = 0; i < pend[kd].size(); i++) {
            const int32_t e = pend[kd][i], k = place_of(pts[e]);
            if (k < 0) continue;
            const int32_t *ptr = kd == 6 ? m.cor_ptr : m.neu_ptr, *cl = kd == 6 ? m.cor_col : m.neu_col;
            sweeps[e] = 1;
            for (int a = ptr[k]; a < ptr[k + 1]; a++) enter(cl[a]);
          }
      for (int s = nu; s >= 1; s--)
        for (int j = 4; j >= 0; j--) {
          // rows of this colour met after this step are needed as the sweep before left them
          const int c = backward ? 4 - j : j;
          now.clear();
          now.swap(pend[c]);
          for (int32_t e : now) {
            sweeps[e] = (int8_t)s;
            ent0[e] = (int64_t)ent.size();
            const int32_t p = pts[e];
            const int64_t base = m.cptr[p >> 6] + (p & 63);
            for (int k = 0; k < m.deg[p]; k++) {
              const int32_t i = enter(m.col[base + (int64_t)k * 64]);
              ent.push_back(i);
            }
          }
        }
      // the list: colours (own, then by sweeps), edge points, corners, read-only points
      PatchDesc D{};
      const int n = (int)pts.size();
      if (n > 65535) {
        bad[t] = 1;
        break;
      }
      auto rank = [&](int e) {      // group of an entry
        const int kd = kind[pts[e]];
        const bool own = e < nown;
        if (kd < 5) return sweeps[e] ? kd * 3 + (own ? 0 : 3 - sweeps[e]) : 19;
        if (sweeps[e] || own) return 15 + (kd - 5) * 2 + (own ? 0 : 1);
        return 19;
      };
      int cntg[20] = {0}, at[20];
      group.resize(n);
      for (int e = 0; e < n; e++) cntg[group[e] = (uint8_t)rank(e)]++;
      for (int g = 0, s = 0; g < 20; g++) {
        at[g] = s;
        s += cntg[g];
      }
      for (int c = 0; c < 5; c++) {
        D.g[c] = at[3 * c];
        D.own[c] = cntg[3 * c];
        D.cnt[c][1] = cntg[3 * c] + (nu == 2 ? cntg[3 * c + 1] : 0);
        D.cnt[c][0] = cntg[3 * c] + cntg[3 * c + 1] + cntg[3 * c + 2];
        H.max_group = std::max(H.max_group, D.cnt[c][0]);
      }
      if (H.max_group > group_max) {
        bad[t] = 1;
        break;
      }
      D.ncs = at[15];
      D.own_e = cntg[15];
      D.ne = cntg[15] + cntg[16];
      D.own_k = cntg[17];
      D.nk = cntg[17] + cntg[18];
      D.nlist = n;
      D.list = (int32_t)H.rows.size();
      D.comp = (int32_t)H.sbase.size();
      D.ov = (int32_t)H.ov_e.size();
      D.nptr = (int32_t)H.nptr.size();
      loc.resize(n);
      H.rows.resize(D.list + n);
      // as met: the own rows first, in ascending order inside a colour (contiguous), as the Hilbert order has them
      for (int e = 0; e < n; e++) loc[e] = at[group[e]]++;
      std::vector<int32_t> &inv = now;   // list position -> entry
      inv.resize(n);
      for (int e = 0; e < n; e++) {
        H.rows[D.list + loc[e]] = pts[e];
        inv[loc[e]] = e;
      }
      H.sbase.resize(D.comp + D.ncs);
      H.ovf.resize(D.comp + D.ncs, 0);
      H.lcol.resize(3 * ((size_t)D.comp + D.ncs), 0u);
      uint32_t *lc = H.lcol.data() + 3 * (size_t)D.comp;
      for (int l = 0; l < D.ncs; l++) {
        const int32_t p = H.rows[D.list + l];
        const int64_t base = m.cptr[p >> 6] + (p & 63), e0 = ent0[inv[l]];
        H.sbase[D.comp + l] = (uint32_t)base | ((uint32_t)m.deg[p] << PATCH_BASE_BITS);
        H.ovf[D.comp + l] = (uint16_t)(H.ov_e.size() - D.ov);
        for (int s = 0; s < m.deg[p]; s++) {
          const uint32_t v = (uint32_t)loc[ent[e0 + s]];
          if (s < 6) {
            lc[(size_t)(s / 2) * D.ncs + l] |= v << (16 * (s & 1));
          } else {
            H.ov_e.push_back((uint32_t)(base + (int64_t)s * 64));
            H.ov_c.push_back((uint16_t)v);
          }
        }
      }
      D.nov = (int32_t)H.ov_e.size() - D.ov;
      if (neumann) {
        for (int l = D.ncs; l < D.ncs + D.ne + D.nk; l++) {
          const int32_t p = H.rows[D.list + l], k = place_of(p);
          const bool corner = kind[p] == 6;
          const int32_t *ptr = corner ? m.cor_ptr : m.neu_ptr, *cl = corner ? m.cor_col : m.neu_col;
          H.nptr.push_back((int32_t)H.ncol.size());
          for (int a = ptr[k]; a < ptr[k + 1]; a++) H.ncol.push_back((uint16_t)loc[enter(cl[a])]);
        }
        H.nptr.push_back((int32_t)H.ncol.size());
      }
      H.max_list = std::max(H.max_list, n);
      H.max_ov = std::max(H.max_ov, D.nov);
      H.max_ncs = std::max(H.max_ncs, D.ncs);
      H.max_neu = std::max(H.max_neu, D.ne + D.nk);
      if (neumann) H.max_ncol = std::max(H.max_ncol, H.nptr.back() - H.nptr[D.nptr]);
      H.d.push_back(D);
    }
  };
  amg_parts(np, parts, [&](int t, int b0, int b1) {
    // point -> (patch + 1, entry of its list); zero pages until a point is met
    uint64_t *where = static_cast<uint64_t *>(std::calloc((size_t)nA, sizeof(uint64_t)));
    try {
      if (where) walk(t, b0, b1, where);
      else bad[t] = 1;
    } catch (const std::bad_alloc &) {
      bad[t] = 1;
    }
    std::free(where);
  });
  size_t list = 0, comp = 0, ov = 0, nptr = 0, ncol = 0;
  for (int t = 0; t < parts; t++) {
    PatchHost &H = part[t];
    if (bad[t]) return false;
    for (PatchDesc &D : H.d) {
      D.list += (int32_t)list;
      D.comp += (int32_t)comp;
      D.ov += (int32_t)ov;
      D.nptr += (int32_t)nptr;
    }
    for (int32_t &x : H.nptr) x += (int32_t)ncol;
    list += H.rows.size();
    comp += H.sbase.size();
    ov += H.ov_e.size();
    nptr += H.nptr.size();
    ncol += H.ncol.size();
  }
  return 3 * comp < (size_t)INT32_MAX && list < (size_t)INT32_MAX;
}

// Marks (by the sign bit of rows) the own points that another patch reads
// without computing them: the values the patches exchange between sweeps.
inline void patch_mark_shared(int nA, std::vector<PatchHost> &part) {
  std::vector<uint8_t> read(nA, 0);
  auto each = [&](auto f) {
    size_t list0 = 0;                // rows before this part
    for (PatchHost &H : part) {
      for (const PatchDesc &d : H.d) f(H.rows.data() + (d.list - list0), d);
      list0 += H.rows.size();
    }
  };
  each([&](int32_t *rows, const PatchDesc &d) {
    for (int i = d.ncs + d.ne + d.nk; i < d.nlist; i++) read[rows[i]] = 1;
  });
  each([&](int32_t *rows, const PatchDesc &d) {
    auto mark = [&](int first, int n) {
      for (int i = first; i < first + n; i++)
        if (read[rows[i]]) rows[i] |= INT32_MIN;
    };
    for (int c = 0; c < 5; c++) mark(d.g[c], d.own[c]);
    mark(d.ncs, d.own_e);
    mark(d.ncs + d.ne, d.own_k);
  });
}

}  // namespace ufe
