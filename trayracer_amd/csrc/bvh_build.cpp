// Binned-SAH BVH builder (host side). See bvh_build.h.
#include "bvh_build.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <future>
#include <limits>
#include <thread>

namespace trt {
namespace {

struct Box {
  float lo[3], hi[3];
  void reset() {
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::numeric_limits<float>::infinity();
      hi[k] = -std::numeric_limits<float>::infinity();
    }
  }
  void grow(const Box& b) {
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::min(lo[k], b.lo[k]);
      hi[k] = std::max(hi[k], b.hi[k]);
    }
  }
  void grow_pt(const float* p) {
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::min(lo[k], p[k]);
      hi[k] = std::max(hi[k], p[k]);
    }
  }
  double area() const {
    const double dx = double(hi[0]) - lo[0], dy = double(hi[1]) - lo[1], dz = double(hi[2]) - lo[2];
    if (dx < 0 || dy < 0 || dz < 0) return 0.0;
    return 2.0 * (dx * dy + dy * dz + dz * dx);
  }
};

struct Ctx {
  const float* box;  // 6 per prim
  std::vector<float> cen;  // 3 per prim
  std::vector<uint32_t>* order;
  int bins;
  int max_leaf;
  double trav_cost;
  std::atomic<int> threads_left;
};

struct SubTree {
  std::vector<BuildNode> nodes;
  int depth = 0;
};

Box prim_box(const Ctx& c, uint32_t p) {
  Box b;
  std::memcpy(b.lo, c.box + size_t(p) * 6, 12);
  std::memcpy(b.hi, c.box + size_t(p) * 6 + 3, 12);
  return b;
}

// Builds the subtree over order[begin, end) into st.nodes (local indices); returns its
// root's local index.
int build_rec(Ctx& c, uint32_t begin, uint32_t end, SubTree& st, int level);

int make_leaf(Ctx& c, uint32_t begin, uint32_t end, const Box& bb, SubTree& st) {
  BuildNode nd;
  std::memcpy(nd.lo, bb.lo, 12);
  std::memcpy(nd.hi, bb.hi, 12);
  nd.left = nd.right = -1;
  nd.first = begin;
  nd.count = end - begin;
  st.nodes.push_back(nd);
  (void)c;
  return int(st.nodes.size()) - 1;
}

int build_rec(Ctx& c, uint32_t begin, uint32_t end, SubTree& st, int level) {
  std::vector<uint32_t>& ord = *c.order;
  const uint32_t n = end - begin;
  Box bb, cb;
  bb.reset();
  cb.reset();
  for (uint32_t i = begin; i < end; ++i) {
    bb.grow(prim_box(c, ord[i]));
    cb.grow_pt(&c.cen[size_t(ord[i]) * 3]);
  }
  if (n <= 1) return make_leaf(c, begin, end, bb, st);

  // binned SAH over all three axes
  const int B = c.bins;
  double best_cost = std::numeric_limits<double>::infinity();
  int best_axis = -1, best_split = -1;
  std::vector<Box> bin_box(B);
  std::vector<uint32_t> bin_cnt(B);
  std::vector<double> right_area(B);
  std::vector<uint32_t> right_cnt(B);
  for (int axis = 0; axis < 3; ++axis) {
    const float lo = cb.lo[axis], hi = cb.hi[axis];
    if (!(hi > lo)) continue;
    const double scale = double(B) / (double(hi) - double(lo));
    for (int b = 0; b < B; ++b) {
      bin_box[b].reset();
      bin_cnt[b] = 0;
    }
    for (uint32_t i = begin; i < end; ++i) {
      const uint32_t p = ord[i];
      int b = int((double(c.cen[size_t(p) * 3 + axis]) - lo) * scale);
      b = std::min(std::max(b, 0), B - 1);
      bin_box[b].grow(prim_box(c, p));
      bin_cnt[b]++;
    }
    Box acc;
    acc.reset();
    uint32_t cnt = 0;
    for (int b = B - 1; b > 0; --b) {
      acc.grow(bin_box[b]);
      cnt += bin_cnt[b];
      right_area[b] = acc.area();
      right_cnt[b] = cnt;
    }
    acc.reset();
    cnt = 0;
    for (int s = 1; s < B; ++s) {  // split between bin s-1 and s
      acc.grow(bin_box[s - 1]);
      cnt += bin_cnt[s - 1];
      if (cnt == 0 || right_cnt[s] == 0) continue;
      const double cost = acc.area() * cnt + right_area[s] * right_cnt[s];
      if (cost < best_cost) {
        best_cost = cost;
        best_axis = axis;
        best_split = s;
      }
    }
  }
  const double parent_area = bb.area();
  const double leaf_cost = double(n);
  const double split_cost =
      parent_area > 0 ? c.trav_cost + best_cost / parent_area : std::numeric_limits<double>::infinity();
  if (n <= uint32_t(c.max_leaf) && (best_axis < 0 || leaf_cost <= split_cost)) return make_leaf(c, begin, end, bb, st);

  uint32_t mid;
  if (best_axis < 0) {
    mid = begin + n / 2;  // all centroids coincide: split the range in half
  } else {
    const float lo = cb.lo[best_axis], hi = cb.hi[best_axis];
    const double scale = double(B) / (double(hi) - double(lo));
    auto it = std::partition(ord.begin() + begin, ord.begin() + end, [&](uint32_t p) {
      int b = int((double(c.cen[size_t(p) * 3 + best_axis]) - lo) * scale);
      b = std::min(std::max(b, 0), B - 1);
      return b < best_split;
    });
    mid = uint32_t(it - ord.begin());
    if (mid == begin || mid == end) mid = begin + n / 2;
  }

  BuildNode nd;
  std::memcpy(nd.lo, bb.lo, 12);
  std::memcpy(nd.hi, bb.hi, 12);
  nd.first = 0;
  nd.count = 0;
  st.nodes.push_back(nd);
  const int me = int(st.nodes.size()) - 1;

  const bool par = n > 65536 && c.threads_left.fetch_sub(1) > 0;
  if (par) {
    SubTree right_tree;
    auto fut = std::async(std::launch::async, [&]() { return build_rec(c, mid, end, right_tree, level + 1); });
    const int l = build_rec(c, begin, mid, st, level + 1);
    const int r_local = fut.get();
    const int off = int(st.nodes.size());
    for (BuildNode x : right_tree.nodes) {
      if (x.count == 0) {
        x.left += off;
        x.right += off;
      }
      st.nodes.push_back(x);
    }
    st.nodes[me].left = l;
    st.nodes[me].right = r_local + off;
  } else {
    const int l = build_rec(c, begin, mid, st, level + 1);
    const int r = build_rec(c, mid, end, st, level + 1);
    st.nodes[me].left = l;
    st.nodes[me].right = r;
  }
  return me;
}

void finish_stats(BuildResult& r) {
  // depth in internal nodes, SAH cost, leaf count (iterative DFS)
  struct It { int node, d; };
  std::vector<It> stack{{0, 0}};
  const double root_area = [&] {
    Box b;
    std::memcpy(b.lo, r.nodes[0].lo, 12);
    std::memcpy(b.hi, r.nodes[0].hi, 12);
    return b.area();
  }();
  r.depth = 0;
  r.sah_cost = 0;
  r.n_leaves = 0;
  while (!stack.empty()) {
    const It it = stack.back();
    stack.pop_back();
    const BuildNode& nd = r.nodes[size_t(it.node)];
    Box b;
    std::memcpy(b.lo, nd.lo, 12);
    std::memcpy(b.hi, nd.hi, 12);
    const double a = root_area > 0 ? b.area() / root_area : 1.0;
    if (nd.count > 0 || nd.left < 0) {
      r.n_leaves++;
      r.sah_cost += a * nd.count;
      r.depth = std::max(r.depth, it.d);
    } else {
      r.sah_cost += a;
      stack.push_back({nd.left, it.d + 1});
      stack.push_back({nd.right, it.d + 1});
    }
  }
}

struct Poly {
  int n = 0;
  double v[12][3];
};

void clip_plane(const Poly& in, int axis, double c, bool keep_below, Poly& out) {
  out.n = 0;
  for (int i = 0; i < in.n; ++i) {
    const double* a = in.v[i];
    const double* b = in.v[(i + 1) % in.n];
    const double da = keep_below ? c - a[axis] : a[axis] - c;
    const double db = keep_below ? c - b[axis] : b[axis] - c;
    if (da >= 0 && out.n < 12) {
      std::memcpy(out.v[out.n++], a, sizeof(double) * 3);
    }
    if ((da < 0) != (db < 0) && out.n < 12) {
      const double t = da / (da - db);
      double* o = out.v[out.n++];
      for (int k = 0; k < 3; ++k) o[k] = a[k] + t * (b[k] - a[k]);
      o[axis] = c;
    }
  }
}

void poly_box(const Poly& p, double lo[3], double hi[3]) {
  for (int k = 0; k < 3; ++k) {
    lo[k] = 1e300;
    hi[k] = -1e300;
  }
  for (int i = 0; i < p.n; ++i)
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::min(lo[k], p.v[i][k]);
      hi[k] = std::max(hi[k], p.v[i][k]);
    }
}

double box_area(const double lo[3], const double hi[3]) {
  const double dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
  return 2.0 * (dx * dy + dy * dz + dz * dx);
}

void emit_box(const double lo[3], const double hi[3], const float* tlo, const float* thi, uint32_t prim,
              std::vector<float>& box, std::vector<uint32_t>& refs) {
  float b[6];
  for (int k = 0; k < 3; ++k) {
    // outward rounding, clamped to the triangle's own box
    float l = float(lo[k]), h = float(hi[k]);
    if (double(l) > lo[k]) l = std::nextafter(l, -std::numeric_limits<float>::infinity());
    if (double(h) < hi[k]) h = std::nextafter(h, std::numeric_limits<float>::infinity());
    b[k] = std::max(l, tlo[k]);
    b[3 + k] = std::min(h, thi[k]);
  }
  box.insert(box.end(), b, b + 6);
  refs.push_back(prim);
}

void split_rec(const Poly& p, int splits, const float* tlo, const float* thi, uint32_t prim, std::vector<float>& box,
               std::vector<uint32_t>& refs) {
  double lo[3], hi[3];
  poly_box(p, lo, hi);
  if (splits <= 0 || p.n < 3) {
    emit_box(lo, hi, tlo, thi, prim, box, refs);
    return;
  }
  int axis = 0;
  for (int k = 1; k < 3; ++k)
    if (hi[k] - lo[k] > hi[axis] - lo[axis]) axis = k;
  const double c = 0.5 * (lo[axis] + hi[axis]);
  Poly a, b;
  clip_plane(p, axis, c, true, a);
  clip_plane(p, axis, c, false, b);
  if (a.n < 3 || b.n < 3) {
    emit_box(lo, hi, tlo, thi, prim, box, refs);
    return;
  }
  double alo[3], ahi[3], blo[3], bhi[3];
  poly_box(a, alo, ahi);
  poly_box(b, blo, bhi);
  const double aa = box_area(alo, ahi), ab = box_area(blo, bhi);
  const int rest = splits - 1;
  const int sa = aa + ab > 0 ? int(std::lround(rest * aa / (aa + ab))) : rest / 2;
  split_rec(a, sa, tlo, thi, prim, box, refs);
  split_rec(b, rest - sa, tlo, thi, prim, box, refs);
}

}  // namespace

void presplit_triangles(const float* pos, uint32_t n, float beta, std::vector<float>& ref_box,
                        std::vector<uint32_t>& ref_prim) {
  ref_box.clear();
  ref_prim.clear();
  std::vector<double> excess(n);
  double total = 0.0;
  for (uint32_t i = 0; i < n; ++i) {
    const float* p = pos + size_t(i) * 9;
    double lo[3], hi[3];
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::min<double>(p[k], std::min<double>(p[3 + k], p[6 + k]));
      hi[k] = std::max<double>(p[k], std::max<double>(p[3 + k], p[6 + k]));
    }
    const double e1[3] = {double(p[3]) - p[0], double(p[4]) - p[1], double(p[5]) - p[2]};
    const double e2[3] = {double(p[6]) - p[0], double(p[7]) - p[1], double(p[8]) - p[2]};
    const double cx = e1[1] * e2[2] - e1[2] * e2[1], cy = e1[2] * e2[0] - e1[0] * e2[2],
                 cz = e1[0] * e2[1] - e1[1] * e2[0];
    const double tri_area = 0.5 * std::sqrt(cx * cx + cy * cy + cz * cz);
    excess[i] = std::max(0.0, box_area(lo, hi) - 2.0 * tri_area);
    total += excess[i];
  }
  const double budget = double(beta) * n;
  ref_box.reserve(size_t((n + budget) * 6 * 1.05));
  ref_prim.reserve(size_t((n + budget) * 1.05));
  for (uint32_t i = 0; i < n; ++i) {
    const float* p = pos + size_t(i) * 9;
    float tlo[3], thi[3];
    for (int k = 0; k < 3; ++k) {
      tlo[k] = std::min(p[k], std::min(p[3 + k], p[6 + k]));
      thi[k] = std::max(p[k], std::max(p[3 + k], p[6 + k]));
    }
    const int splits = total > 0 ? int(budget * excess[i] / total) : 0;
    if (splits == 0) {
      ref_box.insert(ref_box.end(), tlo, tlo + 3);
      ref_box.insert(ref_box.end(), thi, thi + 3);
      ref_prim.push_back(i);
      continue;
    }
    Poly poly;
    poly.n = 3;
    for (int v = 0; v < 3; ++v)
      for (int k = 0; k < 3; ++k) poly.v[v][k] = p[v * 3 + k];
    split_rec(poly, splits, tlo, thi, i, ref_box, ref_prim);
  }
}

BuildResult build_binned_sah(const float* prim_box_data, uint32_t n, int bins, int max_leaf, int n_threads,
                             double trav_cost) {
  BuildResult res;
  res.prim_order.resize(n);
  for (uint32_t i = 0; i < n; ++i) res.prim_order[i] = i;
  if (n == 0) {
    BuildNode nd{};
    nd.left = nd.right = -1;
    nd.first = 0;
    nd.count = 0;
    res.nodes.push_back(nd);
    res.n_leaves = 1;
    return res;
  }
  Ctx c;
  c.box = prim_box_data;
  c.cen.resize(size_t(n) * 3);
  for (uint32_t i = 0; i < n; ++i)
    for (int k = 0; k < 3; ++k)
      c.cen[size_t(i) * 3 + k] = 0.5f * (prim_box_data[size_t(i) * 6 + k] + prim_box_data[size_t(i) * 6 + 3 + k]);
  c.order = &res.prim_order;
  c.bins = std::max(2, bins);
  c.max_leaf = std::max(1, std::min(7, max_leaf));
  c.trav_cost = trav_cost;
  c.threads_left = std::max(0, n_threads - 1);
  SubTree st;
  st.nodes.reserve(size_t(n) * 2 / std::max(1, c.max_leaf / 2) + 16);
  build_rec(c, 0, n, st, 0);
  res.nodes = std::move(st.nodes);
  finish_stats(res);
  return res;
}

namespace {

// The float nearest to v in the outward direction (down for a lower bound, up for an
// upper one) whose low byte is `byte`; false if none is finite. Stepping outward moves
// the bit pattern by one per step (up for a positive value going up or a negative one
// going down, where the magnitude grows; down otherwise), so the answer is found
// directly unless the steps would cross zero, which the step-by-step walk handles.
bool carry_byte(float v, uint32_t byte, bool upper, float& out) {
  if (std::isfinite(v)) {
    const uint32_t u = f2u(v), sign = u & 0x80000000u, mag = u & 0x7fffffffu;
    const bool grows = (sign == 0u) == upper;  // magnitude grows with each step
    if (grows) {
      const uint32_t m = mag + ((byte - mag) & 0xffu);
      if (m < 0x7f800000u) {
        out = u2f(sign | m);
        return true;
      }
      return false;  // the walk reaches infinity first
    }
    const uint32_t k = (mag - byte) & 0xffu;
    if (k <= mag) {  // k = mag lands on a zero of v's sign, as the walk does
      out = u2f(sign | (mag - k));
      return true;
    }
  }
  float x = v;
  for (int k = 0; k <= 512; ++k) {
    if ((f2u(x) & 0xffu) == byte && std::isfinite(x)) {
      out = x;
      return true;
    }
    x = std::nextafter(x, upper ? HUGE_VALF : -HUGE_VALF);
    if (!std::isfinite(x)) return false;
  }
  return false;
}

}  // namespace

namespace {

// Smallest float not below v.
float float_up(double v) {
  float f = float(v);
  if (double(f) < v) f = std::nextafter(f, HUGE_VALF);
  return f;
}

// Centre and half extent of [lo, hi] as stored (see DevNode48); cb / hb: the low bytes the
// centre and the half extent carry, or -1 for none.
bool centre_half(float lo, float hi, int cb, int hb, float& c, float& h) {
  if (!std::isfinite(lo) || !std::isfinite(hi)) return false;
  c = float(0.5 * (double(lo) + double(hi)));
  if (cb >= 0 && !carry_byte(c, uint32_t(cb), false, c)) return false;
  const double half = std::max(double(hi) - double(c), double(c) - double(lo));
  h = float_up(float_up(half) * (1.0 + kHalfExtentMargin));
  if (!std::isfinite(h)) return false;
  if (hb >= 0 && !carry_byte(h, uint32_t(hb), true, h)) return false;
  return true;
}

}  // namespace

bool pack_nodes(const std::vector<DevNode2>& in, std::vector<DevNode48>& out) {
  static_assert(sizeof(DevNode48) == kNodeBytes, "node size");
  if (in.size() >= kMaxDeviceNodes) return false;
  out.resize(in.size());
  for (size_t i = 0; i < in.size(); ++i) {
    const DevNode2& n = in[i];
    DevNode48& d = out[i];
    const float* xy[2] = {n.r0, n.r1};  // lo.x, hi.x, lo.y, hi.y per child
    float* row[2] = {d.r0, d.r1};
    for (int c = 0; c < 2; ++c) {
      const uint32_t ref = uint32_t(device_child_ref(n.c[c]));
      for (int k = 0; k < 2; ++k) {
        const int cb = int((ref >> (16 * k)) & 0xffu), hb = int((ref >> (16 * k + 8)) & 0xffu);
        if (!centre_half(xy[c][2 * k], xy[c][2 * k + 1], cb, hb, row[c][2 * k], row[c][2 * k + 1])) return false;
      }
      if (!centre_half(n.r2[2 * c], n.r2[2 * c + 1], -1, -1, d.r2[2 * c], d.r2[2 * c + 1])) return false;
    }
  }
  return true;
}

namespace {

// 2^e as a double, e in the normal range.
double exp2_int(int e) {
  const uint64_t u = uint64_t(e + 1023) << 52;
  double d;
  std::memcpy(&d, &u, 8);
  return d;
}

// fp16 bits of v >= 0: to nearest (even), or upward. v < 2^16; below 2^-14 the spacing stays
// that of the subnormals.
uint32_t half_bits(double v, bool up) {
  if (!(v > 0.0)) return 0u;
  uint64_t u;
  std::memcpy(&u, &v, 8);
  const int e = int(u >> 52) - 1022;    // v in [2^(e-1), 2^e)
  const int q = std::max(e - 11, -24);  // exponent of the last place
  const double m = v * exp2_int(-q);
  // r in [0, 2^11]: adding it below the exponent field carries into it where it must
  const uint32_t r = uint32_t(up ? std::ceil(m) : std::nearbyint(m));
  const uint32_t expo = uint32_t(q + 24);
  return expo == 0u ? r : ((expo + 1u) << 10) + (r - 1024u);
}

double half_value(uint32_t h) {
  const int e = int((h >> 10) & 31u);
  const double m = double(h & 1023u);
  return e == 0 ? m * exp2_int(-24) : (1024.0 + m) * exp2_int(e - 25);
}

bool empty_child(int32_t c) { return c < 0 && (~uint32_t(c) & 7u) == 0u; }

void child_bounds(const DevNode2& n, int c, float lo[3], float hi[3]) {
  const float* xy = c ? n.r1 : n.r0;
  lo[0] = xy[0]; hi[0] = xy[1]; lo[1] = xy[2]; hi[1] = xy[3];
  lo[2] = n.r2[2 * c]; hi[2] = n.r2[2 * c + 1];
}

// The up to two coordinates at which the most leaf boxes of a tree, and at least kPlaneBoxes,
// are flat on an axis, of up to kPlaneNodes of its nodes taken evenly.
constexpr size_t kPlaneNodes = 16384, kPlaneBoxes = 32;
int flat_planes(const std::vector<DevNode2>& in, size_t first, size_t count, int axis, double at[2]) {
  std::vector<float> v;
  const size_t step = (count + kPlaneNodes - 1) / kPlaneNodes;
  for (size_t i = 0; i < count; i += step)
    for (int c = 0; c < 2; ++c) {
      const DevNode2& n = in[first + i];
      if (n.c[c] >= 0 || empty_child(n.c[c])) continue;
      float lo[3], hi[3];
      child_bounds(n, c, lo, hi);
      if (lo[axis] == hi[axis]) v.push_back(lo[axis]);
    }
  std::sort(v.begin(), v.end());
  size_t boxes[2] = {kPlaneBoxes - 1, kPlaneBoxes - 1};
  int found = 0;
  for (size_t a = 0, b; a < v.size(); a = b) {
    for (b = a + 1; b < v.size() && v[b] == v[a];) ++b;
    if (b - a <= boxes[1]) continue;
    const int place = b - a > boxes[0] ? 0 : 1;
    if (place == 0) {
      boxes[1] = boxes[0];
      at[1] = at[0];
    }
    boxes[place] = b - a;
    at[place] = v[a];
    found = std::min(2, found + 1);
  }
  return found;
}

}  // namespace

bool pack_nodes32(const std::vector<DevNode2>& in, size_t first, size_t count, NodeSpace& space, DevNode32* out,
                  int n_threads, bool stretch) {
  static_assert(sizeof(DevNode32) == 32, "node size");
  double blo[3] = {HUGE_VAL, HUGE_VAL, HUGE_VAL}, bhi[3] = {-HUGE_VAL, -HUGE_VAL, -HUGE_VAL};
  for (int c = 0; c < 2; ++c) {  // the root's children bound the tree
    if (empty_child(in[first].c[c])) continue;
    float lo[3], hi[3];
    child_bounds(in[first], c, lo, hi);
    for (int k = 0; k < 3; ++k) {
      blo[k] = std::min(blo[k], double(lo[k]));
      bhi[k] = std::max(bhi[k], double(hi[k]));
    }
  }
  double Rk[3], R = 0.0;  // the tree's half sides, and the largest
  for (int k = 0; k < 3; ++k) {
    space.org[k] = blo[k] <= bhi[k] ? float(0.5 * (blo[k] + bhi[k])) : 0.f;
    if (!std::isfinite(space.org[k])) return false;
    Rk[k] = blo[k] <= bhi[k] ? std::max(bhi[k] - space.org[k], space.org[k] - blo[k]) : 0.0;
    R = std::max(R, Rk[k]);
  }
  int e = 0;
  if (R > 0.0) (void)std::frexp(R, &e);
  if (!std::isfinite(R) || e < -60 || e > 60) return false;
  space.scale = float(std::ldexp(1.0, e - 14));
  // the planes with the most flat boxes on each axis, two or one, are put on the grid
  for (int k = 0; k < 3; ++k) {
    space.step[k] = space.scale;
    double at[2], c[2];
    const int n = flat_planes(in, first, count, k, at);
    for (int i = 0; i < n; ++i) {
      const double mid = (at[i] - space.org[k]) / space.scale;
      c[i] = half_value(half_bits(std::fabs(mid), false)) * (mid < 0.0 ? -1.0 : 1.0);
    }
    if (stretch && n == 2 && c[0] != c[1]) {
      const double step = (at[1] - at[0]) / (c[1] - c[0]);
      if (std::fabs(step - space.scale) < kMaxStretch * space.scale) space.step[k] = float(step);
    }
    if (n) space.org[k] = float(at[0] - c[0] * space.step[k]);
  }
  double slack[3];
  for (int k = 0; k < 3; ++k) slack[k] = Rk[k] * std::ldexp(1.0, -19);
  std::atomic<size_t> boxes{0}, coarse{0};
  std::atomic<bool> fits{true};
  // leaf boxes that are flat and yet thick, by axis and stored centre
  std::vector<std::atomic<uint32_t>> flat(2 * count > kMaxThickFlat ? size_t(3) << 16 : 0);
  auto pack_range = [&](size_t begin, size_t end) {
    size_t n_boxes = 0, n_coarse = 0;
    size_t flat_at[3] = {};
    uint32_t flat_run[3] = {};  // boxes at flat_at[axis] not yet counted in `flat`
    auto count_flat = [&](int k, size_t at) {
      if (at != flat_at[k] && flat_run[k]) flat[flat_at[k]] += flat_run[k];
      flat_run[k] = at == flat_at[k] ? flat_run[k] + 1u : 1u;
      flat_at[k] = at;
    };
    for (size_t i = begin; i < end; ++i) {
      const DevNode2& n = in[i];
      DevNode32& d = out[i];
      for (int c = 0; c < 2; ++c) {
        const int32_t ref = n.c[c];
        d.w[4 * c + 3] = uint32_t(ref >= 0 ? ref * int32_t(sizeof(DevNode32)) : ref);
        if (empty_child(ref)) {
          for (int k = 0; k < 3; ++k) d.w[4 * c + k] = 0xfc000000u;  // c = 0, h = -inf
          continue;
        }
        float lo[3], hi[3];
        child_bounds(n, c, lo, hi);
        double exact = 0.0, stored = 0.0;
        for (int k = 0; k < 3; ++k) {
          const double S = space.step[k], mid = (0.5 * (double(lo[k]) + double(hi[k])) - space.org[k]) / S;
          if (!(std::fabs(mid) < 32768.0)) {
            fits = false;
            return;
          }
          const uint32_t cb = half_bits(std::fabs(mid), false) | (mid < 0.0 ? 0x8000u : 0u);
          const double cs = (mid < 0.0 ? -1.0 : 1.0) * half_value(cb & 0x7fffu) * S + space.org[k];
          const double half = std::max(double(hi[k]) - cs, cs - double(lo[k]));
          const double h = (half * (1.0 + kHalfExtentMargin) + slack[k]) / S;
          if (!(h < 65504.0)) {
            fits = false;
            return;
          }
          const uint32_t hb = half_bits(h, true);
          d.w[4 * c + k] = cb | (hb << 16);
          if (!flat.empty() && ref < 0 && lo[k] == hi[k] && half_value(hb) * S > kThinHalf * Rk[k]) count_flat(k, (size_t(k) << 16) + cb);
          exact += 0.5 * (double(hi[k]) - double(lo[k]));
          stored += half_value(hb) * S;
        }
        ++n_boxes;
        n_coarse += stored > kCoarseGrowth * exact ? 1u : 0u;
      }
    }
    boxes += n_boxes;
    coarse += n_coarse;
    for (int k = 0; k < 3; ++k)
      if (flat_run[k]) flat[flat_at[k]] += flat_run[k];
  };
  const size_t n_parts = std::min<size_t>(size_t(std::max(1, n_threads)), count / 16384 + 1);
  auto pack_part = [&](size_t t) { pack_range(first + count * t / n_parts, first + count * (t + 1) / n_parts); };
  std::vector<std::thread> pool;
  size_t started = 1;
  try {
    pool.reserve(n_parts);
    for (; started < n_parts; ++started) pool.emplace_back(pack_part, started);
  } catch (...) {  // no more threads to be had: this one packs the rest
  }
  pack_part(0);
  for (size_t t = started; t < n_parts; ++t) pack_part(t);
  for (std::thread& t : pool) t.join();
  size_t coplanar = 0;
  for (const std::atomic<uint32_t>& n : flat) coplanar += n >= kThickPlane ? n.load() : 0u;
  return fits && coplanar <= kMaxThickFlat && double(coarse) <= kCoarseShare * double(boxes);
}

std::vector<DevNode2> to_device_layout(const BuildResult& b) {
  std::vector<DevNode2> out;
  const BuildNode& root = b.nodes[0];
  auto is_leaf = [&](const BuildNode& nd) { return nd.count > 0 || nd.left < 0; };
  auto fill_child = [&](DevNode2& d, int slot, const BuildNode& ch, int32_t ref) {
    if (slot == 0) {
      d.r0[0] = ch.lo[0]; d.r0[1] = ch.hi[0]; d.r0[2] = ch.lo[1]; d.r0[3] = ch.hi[1];
      d.r2[0] = ch.lo[2]; d.r2[1] = ch.hi[2];
    } else {
      d.r1[0] = ch.lo[0]; d.r1[1] = ch.hi[0]; d.r1[2] = ch.lo[1]; d.r1[3] = ch.hi[1];
      d.r2[2] = ch.lo[2]; d.r2[3] = ch.hi[2];
    }
    d.c[slot] = ref;
  };
  if (is_leaf(root)) {
    DevNode2 d{};
    fill_child(d, 0, root, leaf_code(root.first, root.count));
    BuildNode empty{};
    empty.count = 0;
    fill_child(d, 1, empty, leaf_code(0, 0));
    out.push_back(d);
    return out;
  }
  // depth-first numbering of internal nodes, left child first
  std::vector<int> dev_index(b.nodes.size(), -1);
  std::vector<int> order;
  order.reserve(b.nodes.size() / 2 + 1);
  std::vector<int> stack{0};
  while (!stack.empty()) {
    const int i = stack.back();
    stack.pop_back();
    dev_index[size_t(i)] = int(order.size());
    order.push_back(i);
    const BuildNode& nd = b.nodes[size_t(i)];
    if (!is_leaf(b.nodes[size_t(nd.right)])) stack.push_back(nd.right);
    if (!is_leaf(b.nodes[size_t(nd.left)])) stack.push_back(nd.left);
  }
  out.resize(order.size());
  for (size_t k = 0; k < order.size(); ++k) {
    const BuildNode& nd = b.nodes[size_t(order[k])];
    DevNode2 d{};
    const int ch[2] = {nd.left, nd.right};
    for (int s = 0; s < 2; ++s) {
      const BuildNode& cn = b.nodes[size_t(ch[s])];
      const int32_t ref = is_leaf(cn) ? leaf_code(cn.first, cn.count) : dev_index[size_t(ch[s])];
      fill_child(d, s, cn, ref);
    }
    out[k] = d;
  }
  return out;
}

}  // namespace trt
