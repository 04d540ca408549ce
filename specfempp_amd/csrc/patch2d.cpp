// Host side of the 2-D patches: the partition, its index tables and their
// device copies (see patch2d.hpp).
#include "patch2d.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <future>
#include <numeric>

#include "../../include/specfempp_amd.h"

namespace sfx {

namespace {

int point_cap(int pe) { return pe == PATCH_LARGE ? PatchCap<PATCH_LARGE>::points : PatchCap<PATCH_SMALL>::points; }
int boundary_cap(int pe) {
  return pe == PATCH_LARGE ? PatchCap<PATCH_LARGE>::boundary : PatchCap<PATCH_SMALL>::boundary;
}

// Recursive coordinate bisection of elements [a, b) of `order` down to groups
// of at most pe elements: the longer side is cut nearest its middle between
// two distinct centroid coordinates, so that the groups of a structured grid
// are rectangles.
struct Bisection {
  const std::vector<float> &cx, &cz;
  std::vector<int32_t> &order;
  int pe;
  using Groups = std::vector<std::pair<int, int>>;

  int cut(int a, int b, int want) {
    float lo[2] = {cx[order[a]], cz[order[a]]}, hi[2] = {lo[0], lo[1]};
    for (int i = a; i < b; i++) {
      const float x = cx[order[i]], z = cz[order[i]];
      lo[0] = std::min(lo[0], x), hi[0] = std::max(hi[0], x);
      lo[1] = std::min(lo[1], z), hi[1] = std::max(hi[1], z);
    }
    const int axis = hi[0] - lo[0] >= hi[1] - lo[1] ? 0 : 1;
    const std::vector<float> &c = axis == 0 ? cx : cz;
    const int mid = a + want;
    std::nth_element(order.begin() + a, order.begin() + mid, order.begin() + b,
                     [&](int32_t p, int32_t q) { return c[p] != c[q] ? c[p] < c[q] : p < q; });
    // elements within a rounding error of the middle one's coordinate stay
    // together when that leaves both sides non-empty
    const float v = c[order[mid]], eps = 1e-5f * (hi[axis] - lo[axis]);
    const auto first = order.begin() + a, last = order.begin() + b;
    const int below = static_cast<int>(std::partition(first, last, [&](int32_t e) { return c[e] < v - eps; }) - first);
    const int upto =
        below + static_cast<int>(std::partition(first + below, last, [&](int32_t e) { return c[e] <= v + eps; }) -
                                 (first + below));
    const int n = b - a;
    int k = std::abs(below - want) <= std::abs(upto - want) ? below : upto;
    if (k <= 0 || k >= n) k = below > 0 ? below : upto;
    if (k <= 0 || k >= n) {
      std::nth_element(order.begin() + a, order.begin() + mid, order.begin() + b);
      return mid;
    }
    return a + k;
  }
  // [a, b) into `parts` groups of about equal size, cut again where the
  // rounding to whole columns left one too large; the halves of a large range on
  // up to `threads` host threads
  void split(int a, int b, int parts, Groups &out, int threads) {
    if (parts <= 1 && b - a > pe) parts = 2;
    if (parts <= 1 || b - a <= 1) {
      out.push_back({a, b});
      return;
    }
    const int left = parts / 2;
    const int m = cut(a, b, std::max(1, static_cast<int>(static_cast<int64_t>(b - a) * left / parts)));
    if (threads < 2 || b - a < 2000) {
      split(a, m, left, out, 1);
      split(m, b, parts - left, out, 1);
      return;
    }
    Groups right;
    std::future<void> job = std::async(std::launch::async | std::launch::deferred,
                                       [&] { split(m, b, parts - left, right, threads / 2); });
    split(a, m, left, out, threads - threads / 2);
    job.get();
    out.insert(out.end(), right.begin(), right.end());
  }
};

// FNV-1a over 64-bit words of the values
uint64_t hash_of(const std::vector<uint16_t> &v) {
  uint64_t h = 0xcbf29ce484222325ull ^ v.size();
  for (size_t i = 0; i < v.size(); i += 4) {
    uint64_t w = 0;
    std::memcpy(&w, &v[i], std::min<size_t>(4, v.size() - i) * 2);
    h = (h ^ w) * 0x100000001b3ull;
    h ^= h >> 29;
  }
  return h;
}

}  // namespace

// Small patches while large ones would leave compute units without a
// workgroup.  us a step, small and large (colored, 8 sources, 32 receivers; the
// gather form 0.5 to 4 more, in the same order): 6,400 elements 8.62 and 9.19;
// 16,900 9.63 and 9.61; 23,187 10.58 and 11.19; 30,000 11.88 and 11.30; 39,900
// 12.88 and 12.84; 50,000 15.22 and 14.69; 61,103 20.79 and 20.04; 90,000 24.73
// and 24.15; 160,000 39.03 and 37.34; 250,000 54.43 and 54.75; 490,000 128.1 and
// 113.5.  How many rounds of workgroups a size makes moves both forms alike.
int patch_elements(int64_t nspec) { return nspec > 24000 ? PATCH_LARGE : PATCH_SMALL; }

void add_patches(PatchPlan &plan, const HostAssembly &h, const std::vector<int32_t> &key, bool colored) {
  constexpr int npe = 25;
  const int ns = h.nspec, ng = h.nglob_el, pe = plan.pe;
  const int mesh = static_cast<int>(plan.patch_end.size());
  std::vector<float> cx(ns), cz(ns);
  for (int e = 0; e < ns; e++) {
    cx[e] = h.px2d[static_cast<size_t>(e) * npe + 12];
    cz[e] = h.pz2d[static_cast<size_t>(e) * npe + 12];
  }
  std::vector<int32_t> order(ns);
  std::iota(order.begin(), order.end(), 0);
  Bisection bis{cx, cz, order, pe};
  // the average size to aim at, below the limit so that cuts at whole columns
  // seldom leave a group that must be cut again
  const int target = pe == PATCH_LARGE ? 45 : 22;
  Bisection::Groups groups;
  bis.split(0, ns, (ns + target - 1) / target, groups, 8);

  // colored: the points of each element that have a Stacey term, and all of
  // an element with sources, have one more contribution each
  std::vector<int32_t> src_rank(colored ? ns : 0, -1);
  if (colored)
    for (size_t i = 0; i < h.src_order.size(); i++) {
      int32_t &r = src_rank[h.src_ispec[h.src_order[i]]];
      if (r < 0) r = static_cast<int32_t>(i);
    }
  std::vector<std::vector<uint8_t>> edge(colored ? ns : 0);
  if (colored) {
    for (int32_t q : h.bnd_slot) edge[q / npe].push_back(static_cast<uint8_t>(q % npe));
    for (int e = 0; e < ns; e++) {
      std::sort(edge[e].begin(), edge[e].end());
      edge[e].erase(std::unique(edge[e].begin(), edge[e].end()), edge[e].end());
    }
  }
  // boundary points, and the groups cut again until every one fits the
  // kernel's arrays (compact groups fit at once)
  struct Point {
    int32_t first, last;  // patches that visit it
    int32_t count;        // contributions
    int32_t shared;       // 1: a boundary point; index among a patch's visits
  };
  std::vector<Point> point(ng);
  std::vector<char> shared(ng);
  for (;;) {
    std::fill(point.begin(), point.end(), Point{-1, -1, 0, 0});
    std::vector<int> npt(groups.size(), 0), nbd(groups.size(), 0), extra(groups.size(), 0);
    for (size_t k = 0; k < groups.size(); k++) {
      const int32_t patch = static_cast<int32_t>(k);
      for (int i = groups[k].first; i < groups[k].second; i++) {
        if (colored) extra[k] += static_cast<int>(edge[order[i]].size()) + (src_rank[order[i]] >= 0 ? npe : 0);
        const int32_t *ge = &h.gather[static_cast<size_t>(order[i]) * npe];
        for (int p = 0; p < npe; p++) {
          Point &x = point[ge[p]];
          x.count++;
          if (x.last == patch) continue;
          x.last = patch;
          npt[k]++;
          if (x.first < 0) {
            x.first = patch;
            continue;
          }
          nbd[x.first] += !x.shared;
          x.shared = 1;
          nbd[k]++;
        }
      }
    }
    std::vector<std::pair<int, int>> next;
    for (size_t k = 0; k < groups.size(); k++)
      if (npt[k] > point_cap(pe) || nbd[k] > boundary_cap(pe) || extra[k] > pe * npe) {
        const int m = bis.cut(groups[k].first, groups[k].second, (groups[k].second - groups[k].first) / 2);
        next.push_back({groups[k].first, m});
        next.push_back({m, groups[k].second});
      } else {
        next.push_back(groups[k]);
      }
    if (next.size() == groups.size()) break;
    groups = std::move(next);
  }
  for (int g = 0; g < ng; g++) {
    shared[g] = static_cast<char>(point[g].shared);
    point[g].last = -1;
  }
  if (colored)
    for (int e = 0; e < ns; e++) {
      if (src_rank[e] >= 0)
        for (int p = 0; p < npe; p++) point[h.gather[static_cast<size_t>(e) * npe + p]].count++;
      for (uint8_t p : edge[e]) point[h.gather[static_cast<size_t>(e) * npe + p]].count++;
    }

  // numbering: interior points patch by patch (by number of contributions,
  // then first visit), boundary points by first visit over the patches
  std::vector<int32_t> dev(ng, -1);
  std::vector<int32_t> slot(ns);
  const int b_base = plan.nbnd;
  // per boundary point: its contributions as (key, plan element, point)
  struct Entry {
    int32_t b, key, where;  // where: index into plan.bslot
  };
  std::vector<Entry> entries;
  std::vector<uint16_t> t, cat, bidx;
  std::vector<int> by, at, pos, seg, seg_key, lead;
  std::vector<int32_t> visit;     // points of the patch, in the order of their first visit
  std::vector<uint16_t> visited;  // index into it of each element point
  std::vector<uint16_t> number;   // local number of each
  plan.elem.reserve(plan.elem.size() + ns);
  plan.head.reserve(plan.head.size() + groups.size());
  for (size_t k = 0; k < groups.size(); k++) {
    const auto &gr = groups[k];
    const int32_t patch = static_cast<int32_t>(k);
    std::sort(order.begin() + gr.first, order.begin() + gr.second);
    PatchHead hd{};
    hd.el0 = static_cast<int>(plan.elem.size());
    hd.nel = gr.second - gr.first;
    hd.sim = mesh;
    const int32_t *el = &order[gr.first];
    visit.clear();
    visited.resize(static_cast<size_t>(hd.nel) * npe);
    int n[4] = {0, 0, 0, 0};  // points with one, two and more contributions, boundary points
    auto cls = [](const Point &x) { return x.first < 0 ? 3 : x.count == 1 ? 0 : x.count == 2 ? 1 : 2; };
    for (int i = 0; i < hd.nel; i++) {
      slot[el[i]] = static_cast<int32_t>(plan.elem.size());
      plan.elem.push_back(el[i]);
      const int32_t *ge = &h.gather[static_cast<size_t>(el[i]) * npe];
      for (int p = 0; p < npe; p++) {
        Point &x = point[ge[p]];
        if (x.last != patch) {
          x.last = patch;
          if (shared[ge[p]]) x.first = -1;
          x.shared = static_cast<int32_t>(visit.size());
          visit.push_back(ge[p]);
          n[cls(x)]++;
        }
        visited[static_cast<size_t>(i) * npe + p] = static_cast<uint16_t>(x.shared);
      }
    }
    hd.pt0 = plan.nint;
    hd.n1 = n[0];
    hd.n2 = n[1];
    hd.nint = n[0] + n[1] + n[2];
    hd.nb = n[3];
    hd.b0 = static_cast<int>(plan.bpt.size());
    const int l = static_cast<int>(visit.size());
    number.resize(l);
    int at_cls[4] = {0, hd.n1, hd.n1 + hd.n2, hd.nint};
    for (int v = 0; v < l; v++) {
      const int g = visit[v], c = cls(point[g]);
      number[v] = static_cast<uint16_t>(at_cls[c]++);
      if (c < 3) {
        dev[g] = plan.nint + number[v];
        continue;
      }
      int32_t owner = 0;
      if (dev[g] < 0) {
        dev[g] = plan.nbnd++;
        owner = INT32_MIN;
      }
      plan.bpt.push_back({owner | dev[g], 0, 0, 0});
    }
    plan.nint += hd.nint;
    // 16-bit tables: rows, then the contributions of every local point in key
    // order (cat[at[l] .. at[l + 1]) of local point l)
    t.assign(static_cast<size_t>(hd.nel) * 40, 0);
    for (int i = 0; i < hd.nel; i++)
      for (int p = 0; p < npe; p++)
        t[static_cast<size_t>(i) * 40 + p / 5 * 8 + p % 5] = number[visited[static_cast<size_t>(i) * npe + p]];
    by.resize(hd.nel);
    std::iota(by.begin(), by.end(), 0);
    std::sort(by.begin(), by.end(), [&](int a, int b) { return key[el[a]] != key[el[b]] ? key[el[a]] < key[el[b]] : a < b; });
    seg.clear();
    if (colored)
      for (int i = 0; i < hd.nel; i++)
        for (uint8_t p : edge[el[i]]) {
          seg.push_back(t[static_cast<size_t>(i) * 40 + p / 5 * 8 + p % 5]);
          seg_key.resize(seg.size());
          seg_key[seg.size() - 1] = ns + el[i];
        }
    // sources first (by element, in application order), Stacey terms last
    lead.clear();
    if (colored)
      for (int i = 0; i < hd.nel; i++)
        if (src_rank[el[i]] >= 0) lead.push_back(i);
    std::sort(lead.begin(), lead.end(), [&](int a, int b) { return src_rank[el[a]] < src_rank[el[b]]; });
    const int extra = pe * npe, src0 = extra + static_cast<int>(seg.size());
    // Patches of equal connectivity share their tables.  These follow from the
    // rows, the order of the elements and the additional contributions: a patch
    // for which all of that has been seen takes them as they are.
    std::vector<uint16_t> sig(t);
    sig.insert(sig.end(), by.begin(), by.end());
    for (const auto *v : {&seg, &lead}) {
      sig.push_back(static_cast<uint16_t>(v->size()));
      sig.insert(sig.end(), v->begin(), v->end());
    }
    for (int v : {hd.nel, hd.n1, hd.n2, hd.nint, l}) sig.push_back(static_cast<uint16_t>(v));
    const uint64_t sig_hash = hash_of(sig);
    const PatchPlan::Tables *same = nullptr;
    for (auto it = plan.by_shape.equal_range(sig_hash); it.first != it.second && !same; ++it.first)
      if (plan.tables[it.first->second].sig == sig) same = &plan.tables[it.first->second];
    if (!same) {
      at.assign(l + 1, 0);
      for (int i = 0; i < hd.nel; i++)
        for (int p = 0; p < npe; p++) at[t[static_cast<size_t>(i) * 40 + p / 5 * 8 + p % 5] + 1]++;
      for (int v : seg) at[v + 1]++;
      for (int i : lead)
        for (int p = 0; p < npe; p++) at[t[static_cast<size_t>(i) * 40 + p / 5 * 8 + p % 5] + 1]++;
      for (int i = 0; i < l; i++) at[i + 1] += at[i];
      cat.resize(at[l]);
      pos.assign(at.begin(), at.end() - 1);
      for (size_t i = 0; i < lead.size(); i++)
        for (int p = 0; p < npe; p++)
          cat[pos[t[static_cast<size_t>(lead[i]) * 40 + p / 5 * 8 + p % 5]]++] =
              static_cast<uint16_t>(src0 + i * npe + p);
      for (int i : by)
        for (int p = 0; p < npe; p++)
          cat[pos[t[static_cast<size_t>(i) * 40 + p / 5 * 8 + p % 5]]++] = static_cast<uint16_t>(i * npe + p);
      for (size_t i = 0; i < seg.size(); i++) cat[pos[seg[i]]++] = static_cast<uint16_t>(extra + i);
      PatchPlan::Tables made;
      auto mark = [&] { return static_cast<int>(t.size()); };
      made.enta = mark();
      for (int i = 0; i < hd.nint; i++) t.push_back(cat[at[i]]);
      made.entb = mark();
      for (int i = hd.n1; i < hd.nint; i++) t.push_back(cat[at[i] + 1]);
      made.off3 = mark();
      uint16_t o3 = 0;
      for (int i = hd.n1 + hd.n2; i < hd.nint; i++) {
        t.push_back(o3);
        o3 = static_cast<uint16_t>(o3 + at[i + 1] - at[i] - 2);
      }
      t.push_back(o3);
      made.ent3 = mark();
      for (int i = hd.n1 + hd.n2; i < hd.nint; i++)
        t.insert(t.end(), cat.begin() + at[i] + 2, cat.begin() + at[i + 1]);
      made.bent = mark();
      for (int i = hd.nint; i < l; i++)
        for (int j = at[i]; j < at[i + 1]; j++) {
          t.push_back(cat[j]);
          made.bidx.push_back(static_cast<uint16_t>(i - hd.nint));
        }
      // another order of the elements can give the same tables
      made.size = t.size();
      const uint64_t hash = hash_of(t);
      const PatchPlan::Tables *equal = nullptr;
      for (auto it = plan.by_tables.equal_range(hash); it.first != it.second && !equal; ++it.first) {
        const PatchPlan::Tables &o = plan.tables[it.first->second];
        if (o.enta == made.enta && o.entb == made.entb && o.off3 == made.off3 && o.ent3 == made.ent3 &&
            o.bent == made.bent && o.bidx == made.bidx && o.size == t.size() &&
            std::memcmp(&plan.tab[o.base], t.data(), t.size() * 2) == 0)
          equal = &o;
      }
      const int row = static_cast<int>(plan.tables.size());
      if (equal) {
        made.base = equal->base;
      } else {
        plan.tab.resize((plan.tab.size() + 7) / 8 * 8, 0);  // rows are read 16 bytes at a time
        made.base = static_cast<int>(plan.tab.size());
        plan.tab.insert(plan.tab.end(), t.begin(), t.end());
        plan.by_tables.emplace(hash, row);
      }
      made.sig = std::move(sig);
      plan.tables.push_back(std::move(made));
      plan.by_shape.emplace(sig_hash, row);
      same = &plan.tables.back();
    }
    hd.lidx = same->base;
    hd.enta = same->base + same->enta;
    hd.entb = same->base + same->entb;
    hd.off3 = same->base + same->off3;
    hd.ent3 = same->base + same->ent3;
    hd.bent = same->base + same->bent;
    hd.nbent = static_cast<int>(same->bidx.size());
    hd.be0 = static_cast<int>(plan.bslot.size());
    for (int j = 0; j < hd.nbent; j++) {
      const int c = plan.tab[static_cast<size_t>(hd.bent) + j];
      const int32_t order_key = c < extra  ? key[el[c / npe]]
                                : c < src0 ? seg_key[c - extra]
                                           : src_rank[el[lead[(c - src0) / npe]]] - static_cast<int32_t>(h.src_order.size());
      const int32_t b = plan.bpt[static_cast<size_t>(hd.b0) + same->bidx[j]].b & 0x7fffffff;
      entries.push_back({b, order_key, static_cast<int32_t>(plan.bslot.size())});
      plan.bslot.push_back(0);
    }
    plan.head.push_back(hd);
  }
  if (plan.tab.size() > static_cast<size_t>(INT32_MAX) || plan.bslot.size() > static_cast<size_t>(INT32_MAX))
    throw std::invalid_argument("2-D mesh too large for its patch tables");
  // a boundary point's contributions lie together, in key order
  std::vector<int32_t> off(plan.nbnd - b_base + 1, 0);
  for (const Entry &q : entries) off[q.b - b_base + 1]++;
  for (size_t i = 1; i < off.size(); i++) off[i] += off[i - 1];
  const int32_t s_base = plan.boff.empty() ? 0 : plan.boff.back();
  std::vector<Entry> grouped(entries.size());
  {
    std::vector<int32_t> fill(off.begin(), off.end() - 1);
    for (const Entry &q : entries) grouped[fill[q.b - b_base]++] = q;
  }
  if (plan.boff.empty()) plan.boff.push_back(0);
  for (size_t b = 0; b + 1 < off.size(); b++) {
    for (int32_t i = off[b] + 1; i < off[b + 1]; i++)  // a few entries: insertion
      for (int32_t j = i; j > off[b] && grouped[j].key < grouped[j - 1].key; j--) std::swap(grouped[j], grouped[j - 1]);
    for (int32_t i = off[b]; i < off[b + 1]; i++) plan.bslot[grouped[i].where] = s_base + i;
    plan.boff.push_back(s_base + off[b + 1]);
  }
  // boundary points are told apart until finish_patches knows where they start
  for (int g = 0; g < ng; g++)
    if (shared[g]) dev[g] = -1 - dev[g];
  plan.device_of.push_back(std::move(dev));
  plan.slot_of.push_back(std::move(slot));
  plan.patch_end.push_back(static_cast<int>(plan.head.size()));
}

void finish_patches(PatchPlan &plan) {
  for (PatchPoint &p : plan.bpt) {
    const int b = p.b & 0x7fffffff;
    p.k0 = plan.boff[b];
    p.n = plan.boff[b + 1] - plan.boff[b];
  }
  for (auto &d : plan.device_of)
    for (auto &g : d)
      if (g < 0) g = plan.nint + (-1 - g);
  if (plan.boff.empty()) plan.boff.push_back(0);
  plan.tables = {};
  plan.by_shape = {};
  plan.by_tables = {};
}

void renumber_points(HostAssembly &h, const PatchPlan &plan) {
  const std::vector<int32_t> &dev = plan.device_of[0];
  const int ng = h.nglob_el;
  h.lattice_of = dev;
  for (auto &g : h.gather) g = dev[g];
  for (auto &g : h.bnd_gather) g = dev[g];
  std::vector<float> m(h.mass_inverse.size(), 0.0f);
  for (int c = 0; c < h.ncomp; c++)
    for (int g = 0; g < ng; g++)
      m[static_cast<size_t>(c) * h.nglob_pad + dev[g]] = h.mass_inverse[static_cast<size_t>(c) * h.nglob_pad + g];
  h.mass_inverse = std::move(m);
}

namespace {

struct PlanElement {
  const HostAssembly *h;
  size_t e;  // element of its mesh
};
std::vector<PlanElement> plan_elements(const PatchPlan &plan, const std::vector<const HostAssembly *> &meshes) {
  std::vector<PlanElement> out(plan.elem.size());
  for (const PatchHead &hd : plan.head)
    for (int i = hd.el0; i < hd.el0 + hd.nel; i++) out[i] = {meshes[hd.sim], static_cast<size_t>(plan.elem[i])};
  return out;
}
// Stacey entries of every plan element in (element point, edge) order: CSR
struct Entries {
  std::vector<int32_t> off, q;
  struct Span {
    const int32_t *b, *e;
    const int32_t *begin() const { return b; }
    const int32_t *end() const { return e; }
    size_t size() const { return e - b; }
    int32_t operator[](size_t i) const { return b[i]; }
  };
  Span of(size_t i) const { return {q.data() + off[i], q.data() + off[i + 1]}; }
};
Entries plan_stacey(const PatchPlan &plan, const std::vector<const HostAssembly *> &meshes) {
  Entries out;
  out.off.assign(plan.elem.size() + 1, 0);
  for (size_t m = 0; m < meshes.size(); m++)
    for (int32_t sl : meshes[m]->bnd_slot) out.off[plan.slot_of[m][sl / 25] + 1]++;
  for (size_t i = 0; i < plan.elem.size(); i++) out.off[i + 1] += out.off[i];
  out.q.resize(out.off.back());
  std::vector<int32_t> fill(out.off.begin(), out.off.end() - 1);
  for (size_t m = 0; m < meshes.size(); m++)
    for (size_t q = 0; q < meshes[m]->bnd_slot.size(); q++)
      out.q[fill[plan.slot_of[m][meshes[m]->bnd_slot[q] / 25]]++] = static_cast<int32_t>(q);
  for (const PatchHead &hd : plan.head)
    for (int i = hd.el0; i < hd.el0 + hd.nel; i++)
      if (out.off[i + 1] - out.off[i] > 1)
        std::stable_sort(out.q.begin() + out.off[i], out.q.begin() + out.off[i + 1], [&](int32_t a, int32_t b) {
          return meshes[hd.sim]->bnd_slot[a] < meshes[hd.sim]->bnd_slot[b];
        });
  return out;
}

template <class T> void point_to(const T *&p, const DevBuf<char> &mem, size_t at) {
  p = reinterpret_cast<const T *>(mem.p + at);
}

}  // namespace

void PatchDevice::upload_properties(const PatchPlan &plan, const std::vector<const HostAssembly *> &meshes,
                                    hipStream_t s) {
  const std::vector<PlanElement> el = plan_elements(plan, meshes);
  bool once = true;
  auto same = [](float a, float b) { return std::memcmp(&a, &b, sizeof(float)) == 0; };
  for (const PlanElement &p : el) {
    const float *k = &p.h->kappa[p.e * 25], *m = &p.h->mu[p.e * 25];
    for (int i = 1; i < 25 && once; i++) once = same(k[i], k[0]) && same(m[i], m[0]);
    if (!once) break;
  }
  std::vector<float> km, kv, mv;
  if (once) {
    km.resize(2 * el.size());
    for (size_t i = 0; i < el.size(); i++) {
      km[2 * i] = el[i].h->kappa[el[i].e * 25];
      km[2 * i + 1] = el[i].h->mu[el[i].e * 25];
    }
  } else {
    kv.resize(25 * el.size());
    mv.resize(25 * el.size());
    for (size_t i = 0; i < el.size(); i++) {
      std::memcpy(&kv[25 * i], &el[i].h->kappa[el[i].e * 25], 25 * sizeof(float));
      std::memcpy(&mv[25 * i], &el[i].h->mu[el[i].e * 25], 25 * sizeof(float));
    }
  }
  std::vector<float> n, w, rp, rs;
  const auto st = plan_stacey(plan, meshes);
  for (const PatchHead &hd : plan.head)
    for (int i = hd.el0; i < hd.el0 + hd.nel; i++)
      for (int32_t q : st.of(i)) {
        const HostAssembly &h = *meshes[hd.sim];
        n.push_back(h.bnd_normal[2 * q]);
        n.push_back(h.bnd_normal[2 * q + 1]);
        w.push_back(h.bnd_weight[q]);
        rp.push_back(h.bnd_rho_vp[q]);
        rs.push_back(h.bnd_rho_vs[q]);
      }
  PatchBlob b;
  const size_t o[] = {b.add(km), b.add(kv), b.add(mv), b.add(n), b.add(w), b.add(rp), b.add(rs)};
  props_mem.upload(b.bytes, s);
  SFX_HIP(hipStreamSynchronize(s));
  point_to(t.kmu, props_mem, o[0]);
  point_to(t.kappa, props_mem, o[1]);
  point_to(t.mu, props_mem, o[2]);
  point_to(t.bnormal, props_mem, o[3]);
  point_to(t.bweight, props_mem, o[4]);
  point_to(t.brvp, props_mem, o[5]);
  point_to(t.brvs, props_mem, o[6]);
  if (!once) t.kmu = nullptr;
}

void PatchDevice::upload(const PatchPlan &plan, const std::vector<const HostAssembly *> &meshes,
                         bool sources_by_order, const std::vector<PatchSim> &sims, hipStream_t s) {
  pe = plan.pe;
  t = PatchTables{};
  t.nint = plan.nint;
  t.nbnd = plan.nbnd;
  patch_end = plan.patch_end;
  std::vector<PatchHead> heads = plan.head;
  const std::vector<PlanElement> el = plan_elements(plan, meshes);
  auto local_point = [&](const PatchHead &hd, int le, int p) {
    return static_cast<int>(plan.tab[static_cast<size_t>(hd.lidx) + le * 40 + p / 5 * 8 + p % 5]);
  };
  // sources and receivers of every plan element
  std::vector<std::vector<int32_t>> receivers(plan.elem.size());
  std::vector<int> rec_first;
  std::vector<float> h_rec;
  std::vector<std::vector<int32_t>> src_sequence(meshes.size());  // plan element, id pairs in application order
  int src_base = 0, rec_base = 0;
  for (size_t m = 0; m < meshes.size(); m++) {
    const HostAssembly &h = *meshes[m];
    for (size_t i = 0; i < h.src_order.size(); i++) {
      const int32_t sidx = h.src_order[i];
      src_sequence[m].push_back(plan.slot_of[m][h.src_ispec[sidx]]);
      src_sequence[m].push_back(src_base + (sources_by_order ? static_cast<int32_t>(i) : sidx));
    }
    src_base += h.nsrc;
    for (int r = 0; r < h.nrec; r++) receivers[plan.slot_of[m][h.rec_ispec[r]]].push_back(r);
    rec_first.push_back(rec_base);
    h_rec.insert(h_rec.end(), h.rec_h.begin(), h.rec_h.end());
    rec_base += h.nrec;
  }
  std::vector<int32_t> patch_of(plan.elem.size());
  for (size_t k = 0; k < heads.size(); k++)
    for (int i = heads[k].el0; i < heads[k].el0 + heads[k].nel; i++) patch_of[i] = static_cast<int32_t>(k);
  std::vector<std::vector<int32_t>> src_patch(heads.size());
  for (const auto &seq : src_sequence)
    for (size_t i = 0; i < seq.size(); i += 2) {
      src_patch[patch_of[seq[i]]].push_back(seq[i]);
      src_patch[patch_of[seq[i]]].push_back(seq[i + 1]);
    }
  const auto st = plan_stacey(plan, meshes);
  std::vector<int> v_seg_pt, v_seg_loc, v_seg_off(1, 0), v_src_id, v_rp_of, v_rmap;
  std::vector<int4> v_src_el, v_rec;
  int nentry = 0;
  int nrow = 0;
  rec_end.clear();
  for (size_t k = 0; k < heads.size(); k++) {
    PatchHead &hd = heads[k];
    const HostAssembly &h = *meshes[hd.sim];
    const PatchSim &sm = sims[hd.sim];
    hd.dt = sm.dt, hd.dto2 = sm.dto2, hd.dt2o2 = sm.dt2o2;
    hd.nstep = sm.nstep, hd.nsb = sm.nsb;
    while (static_cast<int>(rec_end.size()) < hd.sim) rec_end.push_back(static_cast<int>(v_rec.size()));
    hd.seg0 = static_cast<int>(v_seg_pt.size());
    hd.src0 = static_cast<int>(v_src_el.size());
    hd.rm0 = -1;
    for (int le = 0; le < hd.nel; le++) {
      const int i = hd.el0 + le;
      for (size_t j = 0; j < st.of(i).size(); j++) {
        const int p = h.bnd_slot[st.of(i)[j]] % 25;
        if (j == 0 || h.bnd_slot[st.of(i)[j - 1]] % 25 != p) {
          if (!v_seg_pt.empty()) v_seg_off.push_back(nentry);
          v_seg_pt.push_back(le * 25 + p);
          v_seg_loc.push_back(local_point(hd, le, p));
        }
        nentry++;
      }
      for (int32_t r : receivers[i]) {
        v_rec.push_back(make_int4(rec_first[hd.sim] + r, r, hd.sim, i));
        if (hd.rm0 < 0) {
          hd.rm0 = static_cast<int>(v_rmap.size());
          v_rmap.resize(v_rmap.size() + hd.nint, -1);
        }
        for (int p = 0; p < 25; p++) {
          const int l = local_point(hd, le, p);
          if (l < hd.nint) {
            int &row = v_rmap[hd.rm0 + l];
            if (row < 0) row = nrow++;
            v_rp_of.push_back(row);
          } else {
            v_rp_of.push_back(-1 - (plan.bpt[hd.b0 + l - hd.nint].b & 0x7fffffff));
          }
        }
      }
    }
    // the patch's sources by element, in application order within each
    for (size_t j = 0; j < src_patch[k].size(); j += 2) {
      const int32_t i = src_patch[k][j];
      bool done = false;
      for (size_t m = 0; m < j; m += 2) done = done || src_patch[k][m] == i;
      if (done) continue;
      const int first = static_cast<int>(v_src_id.size());
      for (size_t m = j; m < src_patch[k].size(); m += 2)
        if (src_patch[k][m] == i) v_src_id.push_back(src_patch[k][m + 1]);
      v_src_el.push_back(make_int4(i - hd.el0, first, static_cast<int>(v_src_id.size()), 0));
    }
    hd.nseg = static_cast<int>(v_seg_pt.size()) - hd.seg0;
    hd.nsrc = static_cast<int>(v_src_el.size()) - hd.src0;
  }
  while (rec_end.size() < meshes.size()) rec_end.push_back(static_cast<int>(v_rec.size()));
  if (!v_seg_pt.empty()) v_seg_off.push_back(nentry);
  std::vector<int> v_rec_row(plan.elem.size());
  for (const PatchHead &hd : heads)
    for (int i = hd.el0; i < hd.el0 + hd.nel; i++) {
      const int none = meshes[hd.sim]->nspec_none;
      v_rec_row[i] = plan.elem[i] >= none ? plan.elem[i] - none : -1;
    }
  PatchBlob b;
  const size_t o_row = b.add(v_rec_row);
  const size_t o_head = b.add(heads), o_tab = b.add(plan.tab), o_sim = b.add(sims), o_bpt = b.add(plan.bpt),
               o_boff = b.add(plan.boff), o_bslot = b.add(plan.bslot), o_segp = b.add(v_seg_pt),
               o_segl = b.add(v_seg_loc), o_sego = b.add(v_seg_off), o_srce = b.add(v_src_el),
               o_srci = b.add(v_src_id), o_rec = b.add(v_rec), o_rech = b.add(h_rec), o_rpof = b.add(v_rp_of),
               o_rmap = b.add(v_rmap);
  t.nrow = nrow;
  // geometry: one record per element, control nodes, or per-point arrays
  bool record = true, c4 = true, c9 = true;
  for (const HostAssembly *h : meshes) {
    record = record && !h->geo2d.empty();
    c4 = c4 && h->ngnod2d == 4;
    c9 = c9 && h->ngnod2d == 9;
  }
  const int mode = record ? GEOM2D_RECORD : c4 ? GEOM2D_CTRL4 : c9 ? GEOM2D_CTRL9 : GEOM2D_POINT;
  auto take = [&](const std::vector<float> HostAssembly::*src_v, size_t width) {
    const size_t at = b.room(el.size() * width * sizeof(float));
    char *to = b.bytes.data() + at;
    for (size_t i = 0; i < el.size(); i++, to += width * sizeof(float))
      std::memcpy(to, (el[i].h->*src_v).data() + el[i].e * width, width * sizeof(float));
    return at;
  };
  size_t o_geo[6] = {0, 0, 0, 0, 0, 0};
  if (mode == GEOM2D_RECORD) {
    o_geo[0] = take(&HostAssembly::geo2d, 8);
  } else if (mode == GEOM2D_POINT) {
    o_geo[0] = take(&HostAssembly::xix, 25);
    o_geo[1] = take(&HostAssembly::xiz, 25);
    o_geo[2] = take(&HostAssembly::gammax, 25);
    o_geo[3] = take(&HostAssembly::gammaz, 25);
    o_geo[4] = take(&HostAssembly::jac, 25);
  } else {
    o_geo[0] = take(&HostAssembly::ctrl2d, 2 * static_cast<size_t>(mode));
    // the four-node form takes a row's xi derivatives and a column's gamma
    // derivatives as constant along it, which they are bit for bit
    const std::vector<float> &ds = meshes[0]->dsh2d;
    if (mode == GEOM2D_CTRL4)
      for (int p = 0; p < 25; p++)
        for (int i = 0; i < 4; i++)
          if (ds[8 * p + i] != ds[8 * (p / 5 * 5) + i] || ds[8 * p + 4 + i] != ds[8 * (p % 5) + 4 + i])
            throw std::logic_error("internal: four-node shape derivatives");
    o_geo[5] = b.add(ds);
  }
  tables_mem.upload(b.bytes, s);
  SFX_HIP(hipStreamSynchronize(s));
  point_to(t.head, tables_mem, o_head);
  point_to(t.tab, tables_mem, o_tab);
  point_to(t.sim, tables_mem, o_sim);
  point_to(t.bpt, tables_mem, o_bpt);
  point_to(t.boff, tables_mem, o_boff);
  point_to(t.bslot, tables_mem, o_bslot);
  point_to(t.seg_pt, tables_mem, o_segp);
  point_to(t.seg_loc, tables_mem, o_segl);
  point_to(t.seg_off, tables_mem, o_sego);
  point_to(t.src_el, tables_mem, o_srce);
  point_to(t.src_id, tables_mem, o_srci);
  point_to(t.rec, tables_mem, o_rec);
  point_to(t.rec_h, tables_mem, o_rech);
  point_to(t.rp_of, tables_mem, o_rpof);
  point_to(t.rmap, tables_mem, o_rmap);
  point_to(t.rec_row, tables_mem, o_row);
  t.geom.mode = mode;
  point_to(mode == GEOM2D_RECORD ? t.geom.record : mode == GEOM2D_POINT ? t.geom.xix : t.geom.ctrl, tables_mem,
           o_geo[0]);
  point_to(t.geom.xiz, tables_mem, o_geo[1]);
  point_to(t.geom.gammax, tables_mem, o_geo[2]);
  point_to(t.geom.gammaz, tables_mem, o_geo[3]);
  point_to(t.geom.jac, tables_mem, o_geo[4]);
  point_to(t.geom.dsh, tables_mem, o_geo[5]);
  upload_properties(plan, meshes, s);
  const size_t nb = t.nbnd, nr = plan.boff.back();
  work.alloc(4 * nb + 4 * nr + 12 * static_cast<size_t>(nrow));
  if (work.n) launch_fill(s, work.p, work.n, 0.0f);
  ub = work.p;
  rb[0] = reinterpret_cast<float2 *>(work.p + 4 * nb);
  rb[1] = rb[0] + nr;
  t.snap = work.p + 4 * nb + 4 * nr;
  SFX_HIP(hipStreamSynchronize(s));
}

}  // namespace sfx
