// Tree over the instances' world boxes (the upper level of the two-level
// acceleration), built on the host: the instance count is small beside the
// triangle count.  Host code only.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "devscene.h"

namespace ashd {

struct HostBox {
  double lo[3], hi[3];
};
inline float refBits(int32_t r) {
  float f;
  std::memcpy(&f, &r, 4);
  return f;
}
inline int32_t bitsRef(float f) {
  int32_t r;
  std::memcpy(&r, &f, 4);
  return r;
}

// A binary tree in the BVH2 node layout (child boxes in the parent, leaf = one
// instance), then opened to 4-wide nodes.
//
// Splits are the best of 31 planes per axis by the surface area heuristic (of
// fewer where a node has fewer than 32 items), so that a box much larger than its
// neighbours (a ground plane under a field of instances) leaves near the root: with
// median splits of the box centres it sat in a deep leaf, and every ancestor of it
// covered the scene.  256 instances of four meshes on a ground quad, 4 spp: 7.04 ->
// 6.37 ms.  Where no plane parts the centres, or the better split would make the
// tree deeper than `levels` more levels allow, the median along the widest axis is
// taken.
//
// Items are moved instead of pointed to, all three axes are binned with one vector
// operation each, and a node of few items gets few bins.  2,304 and 100,000
// instances in a field: 0.8 and 47 ms on a 2.7 GHz Xeon, as long as the median
// splits took (0.9 and 47); with index lists, 32 bins at every node and two
// bin computations per item and axis it was 2.4 and 131.
class TlasBuilder {
 public:
  std::vector<float4> nodes;    // binary, node 0 the root
  std::vector<uint32_t> order;  // the instance of leaf k
  uint32_t depth = 0;           // levels of inner nodes below the root

  // Boxes of `ids`, two or more; no leaf lies deeper than `levels` (2^levels >= ids.size()).
  void build(const std::vector<HostBox>& box, const std::vector<uint32_t>& ids, uint32_t levels) {
    items_.resize(ids.size()), spare_.resize(ids.size());
    for (size_t k = 0; k < ids.size(); ++k) {
      Item& i = items_[k];
      i.box = Box{{0, 0, 0, 0}, {0, 0, 0, 0}};
      for (int a = 0; a < 3; ++a) i.box.lo[a] = outward(box[ids[k]].lo[a], false), i.box.hi[a] = outward(box[ids[k]].hi[a], true);
      i.box.hi[3] = refBits(int32_t(ids[k] | 0x40000000u));
    }
    nodes.reserve(4 * ids.size());
    order.reserve(ids.size());
    Box all;
    (void)node(0, items_.size(), all, 0, levels);
  }

  static float outward(double v, bool up) {
    const float x = float(v);
    if (up ? !(double(x) < v) : !(double(x) > v)) return x;
    if (x == 0.0f) return up ? refBits(1) : refBits(int32_t(0x80000001u));
    return refBits(bitsRef(x) + ((x > 0.0f) == up ? 1 : -1));  // its neighbour on that side
  }

 private:
  typedef float Vec __attribute__((vector_size(16)));
  typedef int32_t IVec __attribute__((vector_size(16)));
  struct Box {
    Vec lo, hi;  // x, y, z; fourth lane unused
  };
  struct Item {
    Box box;
    // In hi's fourth lane, plus 2^30: a normal number, which arithmetic on the unused lane takes at full speed.
    uint32_t id() const { return uint32_t(bitsRef(box.hi[3])) & 0x3fffffffu; }
  };
  static constexpr int kBins = 32;
  std::vector<Item> items_, spare_;

  static Vec vmin(Vec a, Vec b) { return b < a ? b : a; }
  static Vec vmax(Vec a, Vec b) { return a < b ? b : a; }
  static void grow(Box& a, const Box& b) { a.lo = vmin(a.lo, b.lo), a.hi = vmax(a.hi, b.hi); }
  static Box none() { return Box{{INFINITY, INFINITY, INFINITY, 0}, {-INFINITY, -INFINITY, -INFINITY, 0}}; }
  static Vec centre(const Box& b) { return 0.5f * b.lo + 0.5f * b.hi; }
  static float area(const Box& b) {
    const Vec d = b.hi - b.lo;
    return d[0] * d[1] + d[1] * d[2] + d[2] * d[0];
  }

  // Splits items [b, e) at the plane of least cost (box area x count on either side), centres in [clo, chi]; returns
  // the first item of the second part, or b when there is none whose parts fit in trees of levels - 1 levels.
  size_t split(size_t b, size_t e, Vec clo, Vec chi, uint32_t levels) {
    const size_t n = e - b;
    const int bins = n >= 32 ? kBins : n >= 16 ? 16 : n >= 6 ? 8 : 4;
    const double most = levels > 60 ? 1e18 : double(uint64_t(1) << (levels ? levels - 1 : 0));
    Vec scale = {0, 0, 0, 0};
    for (int a = 0; a < 3; ++a) {
      const float w = chi[a] - clo[a];
      if (w > 0.0f && std::isfinite(w)) scale[a] = std::min(float(bins) / w, 3.0e38f);
    }
    const Vec last = Vec{1, 1, 1, 1} * float(bins - 1), zero = {0, 0, 0, 0};
    auto bin = [&](const Box& x) {
      Vec t = (centre(x) - clo) * scale;
      t = t > zero ? t : zero;  // not a number: bin 0
      t = t < last ? t : last;
      return __builtin_convertvector(t, IVec);
    };
    Box hb[3][kBins];
    uint32_t cnt[3][kBins];
    for (int a = 0; a < 3; ++a)
      for (int i = 0; i < bins; ++i) hb[a][i] = none(), cnt[a][i] = 0;
    for (size_t k = b; k < e; ++k) {
      const Box x = items_[k].box;
      const IVec i = bin(x);
      for (int a = 0; a < 3; ++a) grow(hb[a][i[a]], x), ++cnt[a][i[a]];
    }
    float best = INFINITY;
    int bestAx = -1, bestBin = 0;
    for (int a = 0; a < 3; ++a) {
      if (!(scale[a] > 0.0f)) continue;
      float right[kBins];
      uint32_t nRight[kBins], m = 0;
      Box acc = none();
      for (int i = bins - 1; i > 0; --i) {
        if (cnt[a][i]) {
          grow(acc, hb[a][i]);
          m += cnt[a][i];
          right[i] = area(acc) * float(m);
        } else {
          right[i] = i < bins - 1 ? right[i + 1] : 0.0f;
        }
        nRight[i] = m;
      }
      acc = none();
      m = 0;
      for (int i = 1; i < bins; ++i) {
        if (!cnt[a][i - 1]) continue;  // the plane before it has the same parts
        grow(acc, hb[a][i - 1]);
        m += cnt[a][i - 1];
        if (!nRight[i]) break;
        if (double(std::max(m, nRight[i])) > most) continue;
        const float cost = area(acc) * float(m) + right[i];
        if (cost < best) best = cost, bestAx = a, bestBin = i;
      }
    }
    if (bestAx < 0) return b;
    const float origin = clo[bestAx], unit = scale[bestAx], plane = float(bestBin);
    size_t left = b, right = 0;  // without a branch on a coin toss
    for (size_t k = b; k < e; ++k) {
      const Item i = items_[k];
      float lo[4], hi[4];
      std::memcpy(lo, &i.box.lo, sizeof lo), std::memcpy(hi, &i.box.hi, sizeof hi);
      const bool second = (0.5f * lo[bestAx] + 0.5f * hi[bestAx] - origin) * unit >= plane;
      items_[left] = i, spare_[right] = i;
      left += !second, right += second;
    }
    std::copy(spare_.begin(), spare_.begin() + right, items_.begin() + left);
    return left;
  }

  int32_t node(size_t b, size_t e, Box& out, uint32_t level, uint32_t levels) {
    if (e - b == 1) {
      out = items_[b].box;
      order.push_back(items_[b].id());
      return encodeLeaf(uint32_t(order.size() - 1), 1);
    }
    depth = std::max(depth, level + 1);
    const size_t at = nodes.size();
    nodes.resize(at + 4);
    size_t m = b + 1;
    if (e - b > 2) {
      Vec clo = centre(items_[b].box), chi = clo;
      for (size_t k = b + 1; k < e; ++k) {
        const Vec c = centre(items_[k].box);
        clo = vmin(clo, c), chi = vmax(chi, c);
      }
      m = split(b, e, clo, chi, levels);
      if (m == b) {
        int ax = 0;
        for (int a = 1; a < 3; ++a)
          if (chi[a] - clo[a] > chi[ax] - clo[ax]) ax = a;
        m = b + (e - b) / 2;
        std::nth_element(items_.begin() + b, items_.begin() + m, items_.begin() + e, [&](const Item& x, const Item& y) {
          float cx = centre(x.box)[ax], cy = centre(y.box)[ax];
          if (cx != cx) cx = 0.0f;  // not a number
          if (cy != cy) cy = 0.0f;
          return cx < cy || (cx == cy && x.id() < y.id());
        });
      }
    }
    Box L, R;
    const int32_t rl = node(b, m, L, level + 1, levels - 1);
    const int32_t rr = node(m, e, R, level + 1, levels - 1);
    nodes[at + 0] = make_float4(L.lo[0], L.hi[0], L.lo[1], L.hi[1]);
    nodes[at + 1] = make_float4(R.lo[0], R.hi[0], R.lo[1], R.hi[1]);
    nodes[at + 2] = make_float4(L.lo[2], L.hi[2], R.lo[2], R.hi[2]);
    nodes[at + 3] = make_float4(refBits(rl), refBits(rr), 0.f, 0.f);
    grow(L, R);
    out = L;
    return int32_t(at / 4);
  }
};

// The binary TLAS as nodes of up to `width` children in the BLAS's 4-wide
// layout, so that one step of the walk serves both levels: a node opens its
// largest internal child until it is full.  Returns the traversal stack entries
// that the part below node `bin` can need (one less than the children per
// node on a path).
inline uint32_t tlasWide(const std::vector<float4>& bin, int32_t node, uint32_t width, std::vector<float4>& out) {
  struct Kid {
    float lo[3], hi[3];
    int32_t ref;
  } kid[4];
  auto load = [&](int32_t n, Kid& a, Kid& b) {
    const float4 *p = &bin[size_t(n) * 4], x = p[0], y = p[1], z = p[2];
    a = Kid{{x.x, x.z, z.x}, {x.y, x.w, z.y}, bitsRef(p[3].x)};
    b = Kid{{y.x, y.z, z.z}, {y.y, y.w, z.w}, bitsRef(p[3].y)};
  };
  auto internal = [](const Kid& k) { return k.ref >= 0 && k.ref != kEmptyRef; };
  auto area = [](const Kid& k) {
    const double x = double(k.hi[0]) - k.lo[0], y = double(k.hi[1]) - k.lo[1], z = double(k.hi[2]) - k.lo[2];
    return x * y + y * z + z * x;
  };
  load(node, kid[0], kid[1]);
  uint32_t n = 2;
  while (n < width) {
    int pick = -1;
    for (uint32_t k = 0; k < n; ++k)
      if (internal(kid[k]) && (pick < 0 || area(kid[k]) > area(kid[pick]))) pick = int(k);
    if (pick < 0) break;
    load(kid[pick].ref, kid[pick], kid[n]);
    ++n;
  }
  const size_t at = out.size();
  out.resize(at + 8);
  uint32_t below = 0;
  int32_t ref[4];
  for (uint32_t k = 0; k < 4; ++k) {
    if (k >= n) {
      for (int a = 0; a < 3; ++a) kid[k].lo[a] = kid[k].hi[a] = 3.0e38f;
      ref[k] = kEmptyRef;
    } else if (internal(kid[k])) {
      ref[k] = int32_t(out.size() / 8);
      below = std::max(below, tlasWide(bin, kid[k].ref, width, out));
    } else {
      ref[k] = kid[k].ref;
    }
  }
  for (int a = 0; a < 3; ++a) {
    out[at + 2 * a] = make_float4(kid[0].lo[a], kid[1].lo[a], kid[2].lo[a], kid[3].lo[a]);
    out[at + 2 * a + 1] = make_float4(kid[0].hi[a], kid[1].hi[a], kid[2].hi[a], kid[3].hi[a]);
  }
  out[at + 6] = make_float4(refBits(ref[0]), refBits(ref[1]), refBits(ref[2]), refBits(ref[3]));
  out[at + 7] = make_float4(0.f, 0.f, 0.f, 0.f);
  return n - 1 + below;
}

struct Tlas {
  std::vector<float4> nodes;    // 4-wide
  std::vector<uint32_t> order;  // the instance of leaf k
  uint32_t depth = 1;           // levels of the binary tree
  uint32_t need = 0;            // traversal stack entries
  uint32_t width = 4;           // children per node at most
};
// The tree over instances `ids`.  blasNeed: stack entries that the deepest BLAS
// needs; room: entries of the smallest traversal stacks.
inline Tlas buildTlas(const std::vector<HostBox>& box, const std::vector<uint32_t>& ids, uint32_t blasNeed, uint32_t room) {
  Tlas t;
  TlasBuilder b;
  if (ids.size() <= 1) {
    const float far = 3.0e38f;
    float lo[3] = {far, far, far}, hi[3] = {far, far, far};
    if (!ids.empty()) {
      for (int a = 0; a < 3; ++a)
        lo[a] = TlasBuilder::outward(box[ids[0]].lo[a], false), hi[a] = TlasBuilder::outward(box[ids[0]].hi[a], true);
      b.order.push_back(ids[0]);
    }
    b.nodes = {make_float4(lo[0], hi[0], lo[1], hi[1]), make_float4(far, far, far, far), make_float4(lo[2], hi[2], far, far),
               make_float4(refBits(ids.empty() ? kEmptyRef : encodeLeaf(0, 1)), refBits(kEmptyRef), 0.f, 0.f)};
    b.depth = 1;
  } else {
    // levels of the balanced tree, and as many more as fit in the smallest stacks: a tree that fitted there still does,
    // and renders with fixed scratch are refused for no other trees
    uint32_t levels = 0;
    while ((size_t(1) << levels) < ids.size()) ++levels;
    const uint32_t need = levels + 1 + blasNeed;
    if (need < room) levels += std::min<uint32_t>(room - need, 16);
    b.build(box, ids, levels);
  }
  t.depth = b.depth;
  t.nodes.reserve(4 * ids.size() + 8);
  t.need = tlasWide(b.nodes, 0, 4, t.nodes);
  // 4-wide unless that needs larger traversal stacks than the smallest ones and than the binary tree
  if (t.need + blasNeed > std::max(room, t.depth + 1 + blasNeed)) {
    t.nodes.clear();
    t.width = 2;
    t.need = tlasWide(b.nodes, 0, 2, t.nodes);
  }
  t.order = std::move(b.order);
  return t;
}

}  // namespace ashd
