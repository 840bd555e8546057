// Patches: the mesh cut into compact groups of nodes, one per workgroup, for
// the passes that form element terms and sum them per node.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <exception>
#include <system_error>
#include <thread>
#include <utility>
#include <vector>

#include "kernels.h"

namespace adcgpu {

// The host side of DevPatch.  Patches are the leaves of repeated cuts of the
// nodes across the longer side of their bounding box, each cut in two until it
// has at most PATCH_NODES nodes, PATCH_ELEMS elements at them and PATCH_WIN
// nodes of those elements (a single node always does, but for a node of more
// than PATCH_ELEMS elements: `ok` is false then).  Every list of a patch starts
// at a multiple of its longest length, so that a block's first loads need no
// directory.  Compact leaves keep the elements formed by two patches few: a
// fifth more than the mesh has.
struct PatchPlan {
  std::vector<int> win, el;
  std::vector<ushort4> lv;
  std::vector<ushort2> cspan;
  std::vector<uint16_t> code;
  int n = 0, wmax = 0;
  bool ok = true;
};

struct PatchNode {
  float x, y;
  int i;
};

// Where nodes [b, e) are cut: after a multiple of the leaf size, along the
// longer side.  Returns the cut; the nodes are partitioned around it.
inline int patch_cut(std::vector<PatchNode>& v, int b, int e) {
  float x0 = v[b].x, x1 = x0, y0 = v[b].y, y1 = y0;
  for (int k = b + 1; k < e; ++k) {
    x0 = std::min(x0, v[k].x); x1 = std::max(x1, v[k].x);
    y0 = std::min(y0, v[k].y); y1 = std::max(y1, v[k].y);
  }
  const int leaves = std::max(2, (e - b + PATCH_NODES - 1) / PATCH_NODES);
  const int mid = b + (int)((int64_t)(e - b) * (leaves / 2) / leaves);
  if (x1 - x0 >= y1 - y0)
    std::nth_element(v.begin() + b, v.begin() + mid, v.begin() + e,
                     [](const PatchNode& p, const PatchNode& q) {
                       return p.x < q.x || (p.x == q.x && p.i < q.i);
                     });
  else
    std::nth_element(v.begin() + b, v.begin() + mid, v.begin() + e,
                     [](const PatchNode& p, const PatchNode& q) {
                       return p.y < q.y || (p.y == q.y && p.i < q.i);
                     });
  return mid;
}

// The patches of nodes [b0, e0) of v, depth first: neighbouring patches are near
// in the list.
inline void patch_leaves(std::vector<PatchNode>& v, int b0, int e0, int np, int ne,
                         const std::vector<int>& nm, const std::vector<int>& ptr,
                         const std::vector<int>& inc, PatchPlan& P) {
  const size_t guess = (size_t)(e0 - b0) / (PATCH_NODES * 4 / 5) + 16;
  P.win.reserve(guess * PATCH_WIN);
  P.el.reserve(guess * PATCH_ELEMS);
  P.lv.reserve(guess * PATCH_ELEMS);
  P.cspan.reserve(guess * PATCH_NODES);
  P.code.reserve(guess * 3 * PATCH_ELEMS);
  // marks of one leaf: stamp, then position
  std::vector<int> nmark(np, 0), npos(np), emark(ne, 0), epos(ne);
  std::vector<int> node, el, halo;
  int stamp = 0;
  std::vector<std::pair<int, int>> todo{{b0, e0}};
  while (!todo.empty()) {
    const int b = todo.back().first, e = todo.back().second;
    todo.pop_back();
    const int cnt = e - b;
    bool leaf = cnt <= PATCH_NODES;
    if (leaf) {
      ++stamp;
      node.clear();
      el.clear();
      halo.clear();
      for (int k = b; k < e; ++k) node.push_back(v[k].i);
      std::sort(node.begin(), node.end());
      for (int k = 0; k < cnt; ++k) {
        nmark[node[k]] = stamp;
        npos[node[k]] = k;
      }
      for (int i : node)
        for (int p = ptr[i]; p < ptr[i + 1]; ++p) {
          const int q = inc[p] / 3;
          if (emark[q] == stamp) continue;
          emark[q] = stamp;
          el.push_back(q);
          for (int k = 0; k < 3; ++k) {
            const int w = nm[3 * (size_t)q + k];
            if (nmark[w] == stamp) continue;
            nmark[w] = stamp;
            halo.push_back(w);
          }
        }
      leaf = (int)el.size() <= PATCH_ELEMS && cnt + (int)halo.size() <= PATCH_WIN;
      if (cnt == 1 && !leaf) {
        P.ok = false;
        return;
      }
    }
    if (!leaf) {
      const int mid = patch_cut(v, b, e);
      todo.push_back({mid, e});
      todo.push_back({b, mid});
      continue;
    }
    std::sort(el.begin(), el.end());
    std::sort(halo.begin(), halo.end());
    for (size_t k = 0; k < halo.size(); ++k) npos[halo[k]] = cnt + (int)k;
    for (size_t k = 0; k < el.size(); ++k) epos[el[k]] = (int)k;
    const size_t w0 = P.win.size(), q0 = P.el.size(), o0 = P.cspan.size(), c0 = P.code.size();
    P.win.resize(w0 + PATCH_WIN, -1);
    P.el.resize(q0 + PATCH_ELEMS, el.empty() ? 0 : el[0]);
    P.lv.resize(q0 + PATCH_ELEMS, make_ushort4(0, 0, 0, 2));
    P.cspan.resize(o0 + PATCH_NODES, make_ushort2(1, 0));
    P.code.resize(c0 + 3 * PATCH_ELEMS, 0);
    std::copy(node.begin(), node.end(), P.win.begin() + w0);
    std::copy(halo.begin(), halo.end(), P.win.begin() + w0 + cnt);
    std::copy(el.begin(), el.end(), P.el.begin() + q0);
    for (size_t k = 0; k < el.size(); ++k) {
      const int* w = &nm[3 * (size_t)el[k]];
      // the patch of the element's first vertex writes its element fields
      P.lv[q0 + k] = make_ushort4((unsigned short)npos[w[0]], (unsigned short)npos[w[1]],
                                  (unsigned short)npos[w[2]], npos[w[0]] < cnt ? 1 : 0);
    }
    size_t c = c0;
    for (int k = 0; k < cnt; ++k) {
      const size_t from = c;
      for (int p = ptr[node[k]]; p < ptr[node[k] + 1]; ++p)
        P.code[c++] = (uint16_t)((inc[p] % 3) * PATCH_ELEMS + epos[inc[p] / 3]);
      P.cspan[o0 + k] = make_ushort2((unsigned short)(from - c0), (unsigned short)(c - c0));
    }
    P.wmax = std::max(P.wmax, cnt + (int)halo.size());
    ++P.n;
  }
}

// fn(0) .. fn(n-1), a thread each; where no thread can be had, in this one.  An
// exception of any of them is rethrown here.
template <class F>
inline void patch_parallel(size_t n, const F& fn) {
  std::vector<std::exception_ptr> err(n);
  auto run = [&](size_t k) {
    try {
      fn(k);
    } catch (...) {
      err[k] = std::current_exception();
    }
  };
  std::vector<std::thread> th;
  th.reserve(n);
  for (size_t k = 0; k < n; ++k) {
    bool started = false;
    if (n > 1) try {
        th.emplace_back(run, k);
        started = true;
      } catch (const std::system_error&) {
      }
    if (!started) run(k);
  }
  for (auto& t : th) t.join();
  for (auto& e : err)
    if (e) std::rethrow_exception(e);
}

// The plan of a mesh: element vertices nm [ne][3], and the incidence lists of
// the nodes (ptr, inc; codes 3 e + k in ascending element order).  Large meshes
// are cut into up to eight parts planned by a thread each (the plan does not
// depend on the number of threads): 1M nodes take 60 ms, one thread 250 ms.
inline PatchPlan patch_plan(int np, int ne, const std::vector<int>& nm, const std::vector<int>& ptr,
                            const std::vector<int>& inc, const double* x, const double* y) {
  std::vector<PatchNode> v(np);
  for (int i = 0; i < np; ++i)  // coordinates only order the cuts; NaN and infinity as zero
    v[i] = {std::isfinite(x[i]) ? (float)x[i] : 0.0f, std::isfinite(y[i]) ? (float)y[i] : 0.0f, i};
  const int levels = np >= 65536 ? 3 : 0;
  std::vector<int> at{0, np};
  for (int l = 0; l < levels; ++l) {
    std::vector<int> next;
    std::vector<int> mid(at.size() - 1);
    patch_parallel(mid.size(), [&](size_t k) { mid[k] = patch_cut(v, at[k], at[k + 1]); });
    for (size_t k = 0; k + 1 < at.size(); ++k) {
      next.push_back(at[k]);
      next.push_back(mid[k]);
    }
    next.push_back(np);
    at = next;
  }
  std::vector<PatchPlan> part(at.size() - 1);
  patch_parallel(part.size(), [&](size_t k) {
    patch_leaves(v, at[k], at[k + 1], np, ne, nm, ptr, inc, part[k]);
  });
  if (part.size() == 1) return std::move(part[0]);
  PatchPlan P;
  size_t n = 0;
  for (const PatchPlan& p : part) n += (size_t)p.n;
  P.win.reserve(n * PATCH_WIN);
  P.el.reserve(n * PATCH_ELEMS);
  P.lv.reserve(n * PATCH_ELEMS);
  P.cspan.reserve(n * PATCH_NODES);
  P.code.reserve(n * 3 * PATCH_ELEMS);
  for (const PatchPlan& p : part) {
    P.win.insert(P.win.end(), p.win.begin(), p.win.end());
    P.el.insert(P.el.end(), p.el.begin(), p.el.end());
    P.lv.insert(P.lv.end(), p.lv.begin(), p.lv.end());
    P.cspan.insert(P.cspan.end(), p.cspan.begin(), p.cspan.end());
    P.code.insert(P.code.end(), p.code.begin(), p.code.end());
    P.n += p.n;
    P.wmax = std::max(P.wmax, p.wmax);
    P.ok = P.ok && p.ok;
  }
  return P;
}

}  // namespace adcgpu
