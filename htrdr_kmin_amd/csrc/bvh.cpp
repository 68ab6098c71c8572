/*
 * Binned-SAH BVH over the ground triangles (see bvh.h for the layout).
 */
#include "bvh.h"

#include "htgx.h"

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <new>
#include <utility>

#include <omp.h>

namespace htgx {
namespace {

constexpr int kBins = 16;
constexpr uint32_t kLeafMax = 4;

struct Box {
  float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX};
  float hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
  void grow(const float p[3])
  {
    for(int a = 0; a < 3; ++a) { lo[a] = std::min(lo[a], p[a]); hi[a] = std::max(hi[a], p[a]); }
  }
  void grow(const Box& b)
  {
    for(int a = 0; a < 3; ++a) { lo[a] = std::min(lo[a], b.lo[a]); hi[a] = std::max(hi[a], b.hi[a]); }
  }
  float area() const
  {
    const float d0 = hi[0] - lo[0], d1 = hi[1] - lo[1], d2 = hi[2] - lo[2];
    if(!(d0 >= 0 && d1 >= 0 && d2 >= 0)) return 0.f;
    return 2.f * (d0 * d1 + d1 * d2 + d2 * d0);
  }
};

/* Triangles [begin, end) of the order */
struct Range { uint32_t begin, end, depth; };

/* From this many triangles a node's own passes run on all threads, one node at
 * a time; smaller ones go to one thread each, with all that is below them. A
 * pass over 16 k triangles takes some 50 us, a few times what starting it on 16
 * threads costs. Scene set-up with 0.5 M triangles: 90 -> 22 ms on 16 threads. */
constexpr uint32_t kParallel = 1u << 14;

/* The minima, maxima and counts gathered over a range do not depend on the
 * order of its triangles, nor does the partition on the threads: the tree and
 * the order of the triangles are those of one thread. */
struct Builder {
  std::vector<Box> tbox;
  std::vector<float> cent; /* [ntris][3] */
  std::vector<uint32_t> order, swap_lo, swap_hi;

  struct Split {
    int axis = 0, bin = -1;
    float lo = 0, scale = 0;
  };

  struct Bins {
    Box box[kBins];
    uint32_t cnt[kBins] = {0};
    void grow(const Bins& o)
    {
      for(int b = 0; b < kBins; ++b) { box[b].grow(o.box[b]); cnt[b] += o.cnt[b]; }
    }
  };

  struct Boxes {
    Box tris, cents;
    void grow(const Boxes& o) { tris.grow(o.tris); cents.grow(o.cents); }
  };

  void gather(uint32_t begin, uint32_t end, Boxes& out) const
  {
    for(uint32_t i = begin; i < end; ++i) {
      out.tris.grow(tbox[order[i]]);
      out.cents.grow(&cent[3 * (size_t)order[i]]);
    }
  }

  void gather(uint32_t begin, uint32_t end, const Split& s, Bins& out) const
  {
    for(uint32_t i = begin; i < end; ++i) {
      const int b = bin_of(order[i], s);
      out.box[b].grow(tbox[order[i]]);
      out.cnt[b]++;
    }
  }

  /* f(begin, end, part) over [begin, end) in a part per thread, folded */
  template<class T, class F>
  T gather_parallel(uint32_t begin, uint32_t end, F&& f) const
  {
    const uint32_t nt = (uint32_t)std::max(1, omp_get_max_threads()), n = end - begin;
    std::vector<T> part(nt);
    #pragma omp parallel for schedule(static, 1)
    for(int64_t k = 0; k < (int64_t)nt; ++k)
      f(begin + (uint32_t)((uint64_t)n * k / nt), begin + (uint32_t)((uint64_t)n * (k + 1) / nt), part[k]);
    for(uint32_t k = 1; k < nt; ++k) part[0].grow(part[k]);
    return part[0];
  }

  int bin_of(uint32_t t, const Split& s) const
  {
    const int b = (int)((cent[3 * (size_t)t + s.axis] - s.lo) * s.scale);
    return std::min(kBins - 1, std::max(0, b));
  }

  /* std::partition of the order by bin < s.bin, on all threads: the misplaced
   * triangles of the lower part, first to last, change places with those of
   * the upper part, last to first */
  uint32_t partition_parallel(uint32_t begin, uint32_t end, const Split& s)
  {
    const uint32_t nt = (uint32_t)std::max(1, omp_get_max_threads()), n = end - begin;
    const uint32_t step = (n + nt - 1) / nt;
    std::vector<uint32_t> lower(nt + 1, 0), nlo(nt + 1, 0), nhi(nt + 1, 0);
    auto first = [&](uint32_t k) { return begin + (uint32_t)std::min<uint64_t>(n, (uint64_t)k * step); };
    #pragma omp parallel for schedule(static, 1)
    for(int64_t k = 0; k < (int64_t)nt; ++k) {
      uint32_t c = 0;
      for(uint32_t i = first(k); i < first(k + 1); ++i) c += bin_of(order[i], s) < s.bin;
      lower[k + 1] = c;
    }
    for(uint32_t k = 0; k < nt; ++k) lower[k + 1] += lower[k];
    const uint32_t mid = begin + lower[nt];
    for(int pass = 0; pass < 2; ++pass) { /* count the misplaced, then list them */
      #pragma omp parallel for schedule(static, 1)
      for(int64_t k = 0; k < (int64_t)nt; ++k) {
        uint32_t l = pass ? nlo[k] : 0, h = pass ? nhi[k] : 0;
        for(uint32_t i = first(k); i < first(k + 1); ++i) {
          const bool low = bin_of(order[i], s) < s.bin;
          if(i < mid && !low) { if(pass) swap_lo[begin + l] = i; ++l; }
          if(i >= mid && low) { if(pass) swap_hi[begin + h] = i; ++h; }
        }
        if(!pass) { nlo[k + 1] = l; nhi[k + 1] = h; }
      }
      if(!pass) for(uint32_t k = 0; k < nt; ++k) { nlo[k + 1] += nlo[k]; nhi[k + 1] += nhi[k]; }
    }
    const uint32_t ns = nlo[nt];
    #pragma omp parallel for schedule(static)
    for(int64_t i = 0; i < (int64_t)ns; ++i)
      std::swap(order[swap_lo[begin + i]], order[swap_hi[begin + ns - 1 - i]]);
    return mid;
  }

  /* Box of the node over r and, of an inner one, its split: binned SAH on the
   * widest centroid axis, child 0 with the lower centroids. False for a leaf. */
  bool split(const Range& r, bool parallel, BvhNode& node, Range child[2])
  {
    const uint32_t begin = r.begin, end = r.end, n = end - begin;
    Boxes boxes;
    if(parallel)
      boxes = gather_parallel<Boxes>(begin, end, [&](uint32_t b, uint32_t e, Boxes& o) { gather(b, e, o); });
    else
      gather(begin, end, boxes);
    const Box& cb = boxes.cents;
    for(int a = 0; a < 3; ++a) { node.lo[a] = boxes.tris.lo[a]; node.hi[a] = boxes.tris.hi[a]; }
    /* the leaves in depth-first order hold the triangles in the order's */
    node.tris = n <= kLeafMax ? (begin << 3) | n : 0;
    if(node.tris) return false;
    Split s;
    for(int a = 1; a < 3; ++a)
      if(cb.hi[a] - cb.lo[a] > cb.hi[s.axis] - cb.lo[s.axis]) s.axis = a;
    const float ext = cb.hi[s.axis] - cb.lo[s.axis];
    uint32_t mid = begin + n / 2;
    if(ext > 0.f) {
      s.lo = cb.lo[s.axis];
      s.scale = (float)kBins / ext;
      Bins bins;
      if(parallel)
        bins = gather_parallel<Bins>(begin, end, [&](uint32_t b, uint32_t e, Bins& o) { gather(b, e, s, o); });
      else
        gather(begin, end, s, bins);
      float right_area[kBins];
      uint32_t right_cnt[kBins];
      Box acc;
      uint32_t c = 0;
      for(int b = kBins - 1; b > 0; --b) {
        acc.grow(bins.box[b]);
        c += bins.cnt[b];
        right_area[b] = acc.area();
        right_cnt[b] = c;
      }
      Box left;
      uint32_t lc = 0;
      float best = FLT_MAX;
      for(int b = 1; b < kBins; ++b) {
        left.grow(bins.box[b - 1]);
        lc += bins.cnt[b - 1];
        if(!lc || !right_cnt[b]) continue;
        const float cost = left.area() * (float)lc + right_area[b] * (float)right_cnt[b];
        if(cost < best) { best = cost; s.bin = b; }
      }
      if(s.bin > 0 && parallel) {
        mid = partition_parallel(begin, end, s);
      } else if(s.bin > 0) {
        const auto it = std::partition(order.begin() + begin, order.begin() + end,
                                       [&](uint32_t t) { return bin_of(t, s) < s.bin; });
        mid = (uint32_t)(it - order.begin());
      }
    }
    if(mid == begin || mid == end) {
      /* all centroids in one bin: split at the median */
      mid = begin + n / 2;
      std::nth_element(order.begin() + begin, order.begin() + mid, order.begin() + end,
                       [&](uint32_t x, uint32_t y) {
                         const float cx = cent[3 * (size_t)x + s.axis], cy = cent[3 * (size_t)y + s.axis];
                         return cx < cy || (cx == cy && x < y);
                       });
    }
    child[0] = Range{begin, mid, r.depth + 1};
    child[1] = Range{mid, end, r.depth + 1};
    return true;
  }

  /* A subtree on one thread, its nodes depth first; the greatest depth below */
  uint32_t build(const Range& r, std::vector<BvhNode>& nodes)
  {
    const size_t idx = nodes.size();
    BvhNode node;
    Range child[2];
    const bool inner = split(r, false, node, child);
    nodes.push_back(node);
    uint32_t depth = r.depth;
    if(inner) {
      const uint32_t d0 = build(child[0], nodes), d1 = build(child[1], nodes);
      depth = std::max(d0, d1);
    }
    nodes[idx].skip = (uint32_t)nodes.size(); /* the first node after the subtree */
    return depth;
  }
};

/* A node built on all threads, or the subtree below one built on one */
struct Top {
  Range r;
  BvhNode node;
  uint32_t child;              /* the first of the two; 0: a subtree */
  std::vector<BvhNode> nodes;  /* of a subtree */
  uint32_t count, first;       /* nodes of all below, place of the first */
};

int build_tree(const float* verts, uint32_t nverts, const uint32_t* tris, const uint32_t* tri_mtl,
               uint32_t ntris, BvhHost& out)
{
  Builder b;
  b.tbox.resize(ntris);
  b.cent.resize(3 * (size_t)ntris);
  b.order.resize(ntris);
  b.swap_lo.resize(ntris);
  b.swap_hi.resize(ntris);
  Box scene;
  bool valid = true;
  #pragma omp parallel if(ntris >= kParallel)
  {
    Box mine;
    bool ok = true;
    #pragma omp for schedule(static) nowait
    for(int64_t t = 0; t < (int64_t)ntris; ++t) {
      for(int k = 0; k < 3; ++k) {
        const uint32_t v = tris[3 * (size_t)t + k];
        if(v >= nverts) { ok = false; continue; }
        b.tbox[t].grow(verts + 3 * (size_t)v);
      }
      for(int a = 0; a < 3; ++a) b.cent[3 * (size_t)t + a] = 0.5f * (b.tbox[t].lo[a] + b.tbox[t].hi[a]);
      b.order[t] = (uint32_t)t;
      mine.grow(b.tbox[t]);
    }
    #pragma omp critical(bvh_box)
    { scene.grow(mine); valid = valid && ok; }
  }
  if(!valid) return HTGX_BAD_ARG;

  /* the large nodes one after the other, then the subtrees below them */
  std::vector<Top> tops(1);
  tops[0].r = Range{0, ntris, 0};
  const bool threads = omp_get_max_threads() > 1;
  for(size_t i = 0; i < tops.size(); ++i) {
    const Range r = tops[i].r;
    tops[i].child = 0;
    if(!threads || r.end - r.begin < kParallel) continue;
    Range child[2];
    b.split(r, true, tops[i].node, child);
    tops[i].child = (uint32_t)tops.size();
    tops.resize(tops.size() + 2);
    for(int k = 0; k < 2; ++k) tops[tops[i].child + k].r = child[k];
  }
  uint32_t depth = 0;
  std::atomic<bool> nomem{false};
  #pragma omp parallel for schedule(dynamic, 1) reduction(max : depth)
  for(int64_t i = 0; i < (int64_t)tops.size(); ++i) {
    if(tops[i].child) continue;
    uint32_t d = 0;
    try { d = b.build(tops[i].r, tops[i].nodes); }
    catch(const std::bad_alloc&) { nomem.store(true); } /* it must not leave the thread's loop */
    depth = std::max(depth, d);
    tops[i].count = (uint32_t)tops[i].nodes.size();
  }
  if(nomem.load()) return HTGX_MEM_ERR;
  out.depth = std::max(out.depth, depth);

  /* depth-first layout: the places of the subtrees, then their nodes */
  for(size_t i = tops.size(); i-- > 0;) /* children follow their parents */
    if(tops[i].child) tops[i].count = 1 + tops[tops[i].child].count + tops[tops[i].child + 1].count;
  out.nodes.clear();
  out.nodes.resize(tops[0].count);
  tops[0].first = 0;
  for(Top& t : tops) {
    if(!t.child) continue;
    t.node.skip = t.first + t.count;
    out.nodes[t.first] = t.node;
    tops[t.child].first = t.first + 1;
    tops[t.child + 1].first = t.first + 1 + tops[t.child].count;
  }
  #pragma omp parallel for schedule(dynamic, 1)
  for(int64_t i = 0; i < (int64_t)tops.size(); ++i) {
    if(tops[i].child) continue;
    BvhNode* to = out.nodes.data() + tops[i].first;
    for(const BvhNode& n : tops[i].nodes) {
      *to = n;
      to++->skip += tops[i].first;
    }
  }
  out.tris.resize(ntris);
  out.prim.assign(b.order.begin(), b.order.end());
  out.mtl.resize(ntris);
  #pragma omp parallel for schedule(static) if(ntris >= kParallel)
  for(int64_t i = 0; i < (int64_t)ntris; ++i) {
    const uint32_t t = b.order[i];
    const float* v0 = verts + 3 * (size_t)tris[3 * (size_t)t + 0];
    const float* v1 = verts + 3 * (size_t)tris[3 * (size_t)t + 1];
    const float* v2 = verts + 3 * (size_t)tris[3 * (size_t)t + 2];
    BvhTri& tr = out.tris[i];
    for(int a = 0; a < 3; ++a) {
      tr.v0[a] = v0[a];
      tr.e1[a] = v1[a] - v0[a];
      tr.e2[a] = v2[a] - v0[a];
    }
    out.mtl[i] = tri_mtl ? tri_mtl[t] : 0u;
  }
  for(int a = 0; a < 3; ++a) { out.lo[a] = scene.lo[a]; out.hi[a] = scene.hi[a]; }
  return HTGX_OK;
}

} /* namespace */

int bvh_build(const float* verts, uint32_t nverts, const uint32_t* tris, const uint32_t* tri_mtl,
              uint32_t ntris, BvhHost& out)
{
  if(!verts || !tris || !nverts || !ntris) return HTGX_BAD_ARG;
  if(ntris >= (1u << 29)) return HTGX_BAD_ARG;
  try { return build_tree(verts, nverts, tris, tri_mtl, ntris, out); }
  catch(const std::bad_alloc&) { return HTGX_MEM_ERR; }
}

} /* namespace htgx */
