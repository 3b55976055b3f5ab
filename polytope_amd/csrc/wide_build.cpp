// Host builder of the four-wide form (WideNode, WideFace, WideLeaf in
// ptx_internal.h; why it visits the reference's leaves is in wide.h).
//
// Which binary nodes a wide node absorbs does not change what is visited, only
// how many nodes a ray reads.  The cut is the one with the least expected
// number of wide nodes a random ray enters, i.e. the least sum of their
// surface areas (the dynamic program of Ylitalo, Karras and Laine, "Efficient
// incoherent ray traversal on GPUs through compressed wide BVHs", 2017, with
// leaves kept as they are): on 1.3 M faces 301,030 nodes with 3.58 children
// each and 12.4 of them on an incoherent ray's way, against 353,856, 3.20 and
// 12.6 for opening the largest child first, and 25.0 binary nodes.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>

#include "wide_build.h"

namespace ptx {

namespace {

constexpr uint32_t kWide = 4;
constexpr float kLimit = 1e16f;                // kWideLimit of wide.h
constexpr int kStepExponent = 24;              // kWideStep of wide.h
constexpr uint32_t kIndexEnd = 0x1FFFFFFEu;    // leaf indices stay below the reserved references
constexpr uint32_t kMaxNodes = 1u << 26;       // 32-bit byte offsets into the node array
// Nodes that a thread checks or builds at least: about 0.1 ms of either.
constexpr size_t kCheckNodes = 8192, kBuildNodes = 2048;
constexpr uint32_t kLeafHeader = kLeafBit, kLeafOne = kLeafBit | (1u << 29), kLeafTwo = kLeafBit | (2u << 29);

// later[] bits of a pair of children i < j (tree order) whose paths part at a
// node split on axis a: octants with a clear visit j after i, the others i
// after j (octants 0-3 have z clear).
struct PairTable {
   uint64_t bits[3][kWide][kWide];                // later[0] in the low 16 bits
   PairTable() {
      std::memset(bits, 0, sizeof(bits));
      for (uint32_t a = 0; a < 3; a++)
         for (uint32_t i = 0; i < kWide; i++)
            for (uint32_t j = i + 1; j < kWide; j++)
               for (uint32_t o = 0; o < 4; o++)
                  bits[a][i][j] |= uint64_t((o >> a & 1u) ? 1u << (4 * j + i) : 1u << (4 * i + j)) << (16 * o);
   }
};

// a - b rounded down or up (Knuth's two-sum gives the rounding error's sign).
double diff(double a, double b, bool up) {
   const double s = a - b, t = s - a;
   const double err = (a - (s - t)) + (-b - t);
   if (up ? err > 0 : err < 0) return std::nextafter(s, up ? INFINITY : -INFINITY);
   return s;
}

// Three of a point's coordinates and whatever follows them in memory.
typedef float Lanes __attribute__((vector_size(16)));
typedef int Mask __attribute__((vector_size(16)));
inline Lanes lanes(const float *p) {
   Lanes x;
   std::memcpy(&x, p, sizeof x);
   return x;
}
inline bool all3(Mask m) { return (m[0] & m[1] & m[2]) != 0; }
inline bool any3(Mask m) { return (m[0] | m[1] | m[2]) != 0; }

// Whether the corners of leaf b's kFaces faces (v, and four bytes behind) span
// its box exactly, none of them NaN (those a minimum skips).
template <int kFaces>
bool corners_span(const ptx_bvh_node &b, const float *v) {
   Lanes lo = lanes(v), hi = lo;
   Mask ok = lo == lo;
   for (int i = 1; i < 3 * kFaces; i++) {
      const Lanes x = lanes(v + 3 * i);
      lo = x < lo ? x : lo;
      hi = x > hi ? x : hi;
      ok &= x == x;
   }
   return all3(ok & (lo == lanes(b.p0)) & (hi == lanes(b.p1)));
}

// WideFace::flat of every face: down the tree, a box that is flat in an axis
// takes its parent's answer if that is flat too, else whether the parent holds
// the coordinate strictly inside.  False when two boxes above one leaf, or two
// leaves of one face, give different answers (trees a caller brings).
bool flat_leaves(const std::vector<ptx_bvh_node> &nodes, size_t faces, UnsetVector<uint8_t> &out) {
   constexpr uint8_t kNot = 0xFF;
   std::vector<uint8_t> inside(nodes.size(), kNot);
   inside[0] = 7;
   out.assign(faces, kNot);
   bool same = true;
   for (size_t i = 0; i < nodes.size(); i++) {
      const ptx_bvh_node &b = nodes[i];
      if (inside[i] == kNot) continue;          // a node that nothing refers to
      if (b.num_faces) {
         uint8_t axes = 0;
         for (int a = 0; a < 3; a++) axes |= b.p0[a] == b.p1[a] ? inside[i] & 1u << a : 0u;
         uint8_t &f = out[b.offset];
         same &= f == kNot || f == axes;
         f = axes;
         continue;
      }
      for (const size_t c : {i + 1, i + b.offset}) {
         uint8_t in = 0;
         for (int a = 0; a < 3; a++) {
            const float x = nodes[c].p0[a];
            if (x == nodes[c].p1[a] && (b.p0[a] == b.p1[a] ? inside[i] >> a & 1u : b.p0[a] < x && x < b.p1[a]))
               in |= uint8_t(1u << a);
         }
         same &= inside[c] == kNot || inside[c] == in;
         inside[c] = in;
      }
   }
   for (uint8_t &f : out) f = f == kNot ? 0 : f;
   return same;
}

// 2^e for e in the normal range.
double pow2(int e) {
   const uint64_t bits = uint64_t(1023 + e) << 52;
   double x;
   std::memcpy(&x, &bits, 8);
   return x;
}

// floor(log2(x)) of a normal x > 0.
int floor_log2(double x) {
   uint64_t bits;
   std::memcpy(&bits, &x, 8);
   return int(bits >> 52) - 1023;
}

// Subtree costs of the cut: cost[i - 1] = the least area sum when the subtree
// hangs from at most i children slots; split: how many of 4, 3 and 2 slots the
// low child takes (0: the node keeps one slot as a wide node of its own).
struct Cut {
   float cost[3];
   uint8_t split4, split3, split2;
};

// Children of the wide node at binary node q, in tree order; pair(i, j, axis)
// for every two of them with the axis of the node their paths part at.
struct Gather {
   const std::vector<ptx_bvh_node> &nodes;
   const UnsetVector<Cut> &cut;
   uint32_t child[kWide];
   uint32_t n = 0;
   uint8_t axis[kWide][kWide];

   void add(uint32_t x, uint32_t slots) {
      const ptx_bvh_node &b = nodes[x];
      const uint32_t k = b.num_faces || slots == 1 ? 0u : slots == 2 ? cut[x].split2 : cut[x].split3;
      if (k == 0) child[n++] = x;
      else open(x, k, slots);
   }
   void open(uint32_t x, uint32_t k, uint32_t slots) {
      const ptx_bvh_node &b = nodes[x];
      const uint32_t first = n;
      add(x + 1, k);
      const uint32_t mid = n;
      add(x + b.offset, slots - k);
      for (uint32_t i = first; i < mid; i++)
         for (uint32_t j = mid; j < n; j++) axis[i][j] = (uint8_t)b.flags;
   }
   void root(uint32_t q) {
      n = 0;
      open(q, cut[q].split4, kWide);
   }
};

}  // namespace

bool build_wide(const HostBvh &bvh, const HostImage &img, unsigned threads, WideImage &out) {
   out = WideImage{};
   const std::vector<ptx_bvh_node> &nodes = bvh.nodes;
   const size_t nn = nodes.size(), np = bvh.pairs.size() / 2;
   if (nn == 0 || np >= kIndexEnd || nn >= 0x7FFFFFFFu) return false;
   // boxes finite, ordered, below the limit, and inside their parents': what
   // the equality of the leaves visited rests on.  In the same pass, which
   // leaves need no header: of one or two faces whose corners span the box.
   UnsetVector<uint8_t> plain(nn);
   std::atomic<bool> nest{true}, flat{false};
   auto check = [&](size_t lo, size_t hi) {
      bool good = true, some = false;
      for (size_t i = lo; i < hi && good; i++) {
         const ptx_bvh_node &b = nodes[i];
         const Lanes p0 = lanes(b.p0), p1 = lanes(b.p1);
         good &= all3((p0 <= p1) & (p0 > -kLimit) & (p1 < kLimit));
         if (b.num_faces) {
            some |= any3(p0 == p1);
            const float *v = &img.tris[9 * size_t(b.offset)];
            plain[i] = b.num_faces == 1 ? corners_span<1>(b, v) : b.num_faces == 2 && corners_span<2>(b, v);
            continue;
         }
         const ptx_bvh_node &l = nodes[i + 1], &h = nodes[i + b.offset];
         good &= all3((lanes(l.p0) >= p0) & (lanes(l.p1) <= p1) & (lanes(h.p0) >= p0) & (lanes(h.p1) <= p1));
      }
      if (!good) nest = false;
      if (some) flat = true;
   };
   // beside it the cut, from the last node to the first (children follow their
   // parents; of boxes that do not nest it is any cut)
   UnsetVector<Cut> cut(nn);
   auto cuts = [&] {
      for (size_t q = nn; q-- > 0;) {
         const ptx_bvh_node &b = nodes[q];
         Cut &c = cut[q];
         if (b.num_faces) {
            c = Cut{{0.f, 0.f, 0.f}, 0, 0, 0};
            continue;
         }
         const Cut &l = cut[q + 1], &r = cut[q + b.offset];
         const float d2 = l.cost[0] + r.cost[0];
         const float d3a = l.cost[0] + r.cost[1], d3b = l.cost[1] + r.cost[0];
         const float d4a = l.cost[0] + r.cost[2], d4b = l.cost[1] + r.cost[1], d4c = l.cost[2] + r.cost[0];
         const float d3 = std::min(d3a, d3b);
         float d4 = d4b;
         c.split4 = 2;
         if (d4a < d4) { d4 = d4a; c.split4 = 1; }
         if (d4c < d4) { d4 = d4c; c.split4 = 3; }
         const float x = b.p1[0] - b.p0[0], y = b.p1[1] - b.p0[1], z = b.p1[2] - b.p0[2];
         c.cost[0] = d4 + (x * y + y * z + z * x);
         c.split3 = c.cost[0] <= d3 ? 0 : d3a <= d3b ? 1 : 2;
         c.split2 = c.cost[0] <= d2 ? 0 : 1;
         c.cost[1] = std::min(c.cost[0], d2);
         c.cost[2] = std::min(c.cost[0], d3);
      }
   };
   host_ranges(nn, threads, kCheckNodes, check, cuts);
   if (!nest) return false;
   if (flat && !flat_leaves(nodes, np, out.flat)) return false;
   // wide nodes in tree order
   UnsetVector<uint32_t> index(nn), roots;
   WideLeaf empty;
   for (int k = 0; k < 3; k++) {
      empty.box[k] = INFINITY;
      empty.box[3 + k] = -INFINITY;
   }
   empty.first = empty.count = 0;
   out.leaves.push_back(empty);
   roots.reserve(nn / 4 + 1);
   std::vector<uint8_t> is_root(nn, 0);
   is_root[0] = 1;
   Gather g{nodes, cut};
   for (size_t q = 0; q < nn; q++) {
      const ptx_bvh_node &b = nodes[q];
      if (!b.num_faces) {
         if (!is_root[q]) continue;
         index[q] = (uint32_t)roots.size();
         roots.push_back((uint32_t)q);
         g.root((uint32_t)q);
         for (uint32_t k = 0; k < g.n; k++) is_root[g.child[k]] = 1;
      } else if (plain[q]) {
         index[q] = (b.num_faces == 1 ? kLeafOne : kLeafTwo) | b.offset;
      } else {
         index[q] = kLeafHeader | (uint32_t)out.leaves.size();
         out.leaves.push_back(
               WideLeaf{{b.p0[0], b.p0[1], b.p0[2], b.p1[0], b.p1[1], b.p1[2]}, b.offset, b.num_faces});
      }
   }
   if (roots.size() > kMaxNodes) return false;
   if (out.leaves.size() >= kIndexEnd) return false;
   static const PairTable pairs;
   out.nodes.resize(roots.size());
   std::vector<uint8_t> count(roots.size());
   host_ranges(roots.size(), threads, kBuildNodes, [&](size_t first, size_t last) {
      Gather g{nodes, cut};
      for (size_t w = first; w < last; w++) {
         g.root(roots[w]);
         const ptx_bvh_node &box = nodes[roots[w]];
         WideNode &o = out.nodes[w];
         for (int a = 0; a < 3; a++) {
            // the children fill their node's box; the least step of which 255
            // reach across it, no smaller than 2^-60 so that its products do
            // not underflow
            const float lo = box.p0[a];
            const double extent = diff(box.p1[a], lo, true);
            int e = -60;
            if (extent > 0) {
               e = std::max(floor_log2(extent / 255.0), -60);
               while (extent * pow2(-e) > 255.0) e++;
            }
            o.org[a] = lo;
            o.exponent[a] = (int8_t)(e + kStepExponent);
            const double inv = pow2(-e);
            for (uint32_t k = 0; k < kWide; k++) {
               uint8_t &p0 = o.planes[2 * a][k], &p1 = o.planes[2 * a + 1][k];
               if (k >= g.n) {
                  p0 = 255;
                  p1 = 0;
                  continue;
               }
               const ptx_bvh_node &c = nodes[g.child[k]];
               const double d0 = diff(c.p0[a], lo, false) * inv, d1 = diff(c.p1[a], lo, true) * inv;
               p0 = (uint8_t)d0;                                 // down
               p1 = (uint8_t)((int)d1 + ((double)(int)d1 < d1));  // up
            }
         }
         o.used = (uint8_t)((1u << g.n) - 1u);
         for (uint32_t k = 0; k < kWide; k++) o.ref[k] = k < g.n ? index[g.child[k]] : kLeafHeader;
         uint64_t later = 0;
         for (uint32_t i = 0; i < g.n; i++)
            for (uint32_t j = i + 1; j < g.n; j++) later |= pairs.bits[g.axis[i][j]][i][j];
         std::memcpy(o.later, &later, sizeof(o.later));
         count[w] = (uint8_t)g.n;
      }
   });
   // deferred stack: a step writes its passing children and pops one of them
   std::vector<uint32_t> depth(roots.size());
   for (size_t w = roots.size(); w-- > 0;) {
      uint32_t below = 0;
      for (uint32_t k = 0; k < count[w]; k++)
         if (!(out.nodes[w].ref[k] & kLeafBit)) below = std::max(below, depth[out.nodes[w].ref[k]]);
      depth[w] = std::max<uint32_t>(count[w], count[w] - 1u + below);
   }
   out.stack = 1u + (roots.empty() ? 0u : depth[0]);      // the sentinel first
   // exact_trace keeps one word per binary level in the same memory
   out.stack = std::max(out.stack, (img.max_stack + 1) / 2);
   out.root = index[0];
   return true;
}

}  // namespace ptx
