// Host check of the four-wide tree form (polytope_amd/csrc/wide.h,
// wide_build.cpp): on random and on grid-aligned scenes, the leaves whose
// faces are tested, their order, the hit and the number of face tests after
// it must be those of the reference's traversal of the binary tree, for every
// ray that is not handed to the binary records.  Rays: random directions,
// components of +0 and -0, origins on box planes, tiny, huge, infinite and NaN
// components.  Prints the numbers of rays and mismatches; exit 1 on a mismatch.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "wide.h"
#include "wide_build.h"

namespace ptx {
int set_error(int code, const std::string &) { return code; }
}  // namespace ptx

using namespace ptx;
using namespace ptx::dev;

struct Seen {
   std::vector<uint32_t> faces;      // faces tested, in order
   float t = INFINITY;
   uint32_t hit = 0xFFFFFFFFu, after = 0;
   bool same(const Seen &o) const {
      return faces == o.faces && hit == o.hit && after == o.after && std::memcmp(&t, &o.t, 4) == 0;
   }
};

// One face, as both traversals test it.
static void face(const HostImage &img, uint32_t k, const Ray &r, Seen &s) {
   float u, v, w;
   s.faces.push_back(k);
   if (test_triangle(&img.tris[9 * size_t(k)], r, s.t, u, v, w, false)) {
      s.hit = k;
      s.after = 0;
   }
   s.after++;
}

// bvh::intersect_compact's order over the compact nodes: pop, test the box
// against the current MinT, push the children.
static Seen binary(const HostBvh &bvh, const HostImage &img, const Ray &r) {
   Seen s;
   std::vector<uint32_t> st = {0};
   while (!st.empty()) {
      const uint32_t i = st.back();
      st.pop_back();
      const ptx_bvh_node &b = bvh.nodes[i];
      float near, far;
      slab(b.p0[0], b.p0[1], b.p0[2], b.p1[0], b.p1[1], b.p1[2], r, near, far);
      if (!(near <= far && near <= s.t)) continue;
      if (b.num_faces) {
         for (uint32_t k = 0; k < b.num_faces; k++) face(img, b.offset + k, r, s);
         continue;
      }
      const uint32_t lo = i + 1, hi = i + b.offset;
      const bool high_first = r.nk >> b.flags & 1u;
      st.push_back(high_first ? lo : hi);
      st.push_back(high_first ? hi : lo);
   }
   return s;
}

// The four-wide traversal; false when the ray goes to the binary records.
static bool wide(const WideImage &w, const HostImage &img, const Ray &r, Seen &s, uint32_t &deepest) {
   if (r.nk & kRayHard) return false;
   float near, far;
   slab(img.root_box[0], img.root_box[1], img.root_box[2], img.root_box[3], img.root_box[4], img.root_box[5], r, near,
        far);
   if (!(near <= far && near <= s.t)) return true;
   struct Entry {
      uint32_t ref;
      float near;
   };
   std::vector<Entry> st(w.stack + 8);
   st[0] = Entry{0xFFFFFFFFu, -INFINITY};      // the sentinel
   uint32_t sp = 1, cur = w.root;
   while (true) {
      if (!(cur & kLeafBit)) {
         const WideNode &n = w.nodes[cur];
         auto word = [&](uint32_t k) {
            uint32_t x;
            std::memcpy(&x, n.planes[k], 4);
            return x;
         };
         const uint32_t x = r.nk & 1u, y = r.nk >> 1 & 1u, z = r.nk >> 2 & 1u;
         const WidePlanes p = {word(x), word(x ^ 1u), word(2 + y), word(2 + (y ^ 1u)), word(4 + z), word(4 + (z ^ 1u))};
         const WideFrame f = wide_frame(r, n.org[0], n.org[1], n.org[2], n.exponent[0], n.exponent[1], n.exponent[2]);
         float nr[4];
         uint32_t m = 0;
         for (int k = 0; k < 4; k++)
            m |= ((r.nk & kRaySlow) ? wide_child_slow(p, k, r, n.org[0], n.org[1], n.org[2], n.exponent[0],
                                                      n.exponent[1], n.exponent[2], s.t, nr[k])
                                    : wide_child(p, k, f, s.t, nr[k]))
                       ? 1u << k
                       : 0u;
         m &= n.used;
         const uint32_t later = n.later[r.nk >> (kRayLaterShift + 4) & 3u] ^ (z ? kLaterFlip : 0u);
         const uint32_t after = later & (m * 0x1111u);
         uint32_t places = 0;
         for (uint32_t k = 0; k < 4; k++)
            if (m >> k & 1u) {
               const uint32_t at = __builtin_popcount(after & (15u << (4 * k)));
               st[sp + at] = Entry{n.ref[k], nr[k]};
               places |= 1u << at;
            }
         if (places != (1u << __builtin_popcount(m)) - 1u) deepest = 0xFFFFFFFFu;   // two children in one place
         sp += __builtin_popcount(m);
         deepest = std::max(deepest, sp);
      } else {
         float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
         const uint32_t kind = cur & ~kWideIndex, idx = cur & kWideIndex;
         uint32_t first = idx, count = kind == kWideOne ? 1 : 2;
         if (kind == kWideHeader) {
            const WideLeaf &l = w.leaves[idx];
            for (int a = 0; a < 3; a++) { lo[a] = l.box[a]; hi[a] = l.box[3 + a]; }
            first = l.first;
            count = l.count;
         } else {
            for (uint32_t k = 0; k < 3 * count; k++)
               for (int a = 0; a < 3; a++) {
                  const float x = img.tris[9 * size_t(first) + 3 * k + a];
                  lo[a] = std::fmin(lo[a], x);
                  hi[a] = std::fmax(hi[a], x);
               }
         }
         slab(lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], r, near, far);
         if (near <= far && near <= s.t && count) {
            if ((r.nk & kRayMinus) && wide_flat(lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], r)) return false;
            for (uint32_t k = 0; k < count; k++) face(img, first + k, r, s);
         }
      }
      do cur = st[--sp].ref;
      while (st[sp].near > wide_bound(s.t));
      if (cur == 0xFFFFFFFFu) return true;
   }
}

int main() {
   std::mt19937 rng(11);
   auto uni = [&](float a, float b) { return a + (b - a) * float(rng() >> 8) * 0x1p-24f; };
   long rays = 0, bad = 0, handed = 0, hits = 0;
   for (int scene = 0; scene < 24; scene++) {
      // random soup, integer-grid boxes' faces, flat sheets, duplicated faces, and one- to three-face scenes
      const int kind = scene % 6;
      const uint32_t nf = kind == 5 ? 1 + scene / 6 : 40u << (scene / 4);
      const float scale = scene % 7 == 3 ? 1e4f : scene % 7 == 5 ? 1e-4f : 1.f;
      WorldMesh m;
      m.nf = nf;
      m.wv.resize(9 * size_t(nf));
      for (uint32_t f = 0; f < nf; f++) {
         const float c[3] = {uni(-4, 4), uni(-4, 4), uni(-4, 4)};
         for (int v = 0; v < 3; v++)
            for (int a = 0; a < 3; a++) {
               float x = c[a] + uni(-0.6f, 0.6f);
               if (kind == 1 || kind == 3) x = std::round(x);
               if (kind == 2 && a == (int)(f % 3)) x = float(int(f % 5) - 2);
               if (kind == 4) x = f % 2 ? m.wv[9 * size_t(f - 1) + 3 * v + a] / scale : std::round(x * 2) * 0.5f;
               m.wv[9 * size_t(f) + 3 * v + a] = x * scale;
            }
      }
      std::vector<WorldMesh> meshes = {m};
      HostBvh bvh;
      build_reference_bvh(meshes, 2, bvh);
      HostImage img;
      WideImage w;
      if (layout_scene(meshes, bvh, img) != PTX_OK || !build_wide(bvh, img, 2, w)) {
         std::printf("scene %d has no wide form\n", scene);
         return 1;
      }
      for (int q = 0; q < 20000; q++) {
         float o[3], d[3];
         for (int a = 0; a < 3; a++) {
            o[a] = uni(-6, 6) * scale;
            d[a] = uni(-1, 1);
            const uint32_t x = rng() % 64;
            if (q % 2) {
               if (x < 16) o[a] = std::round(o[a] / scale) * scale;
               if (x == 17) o[a] = -0.f;
               if (x == 18) o[a] = m.wv[rng() % m.wv.size()];
               if (x >= 20 && x < 30) d[a] = 0.f;
               if (x >= 30 && x < 40) d[a] = -0.f;
               if (x == 40) d[a] = 1e-39f;
               if (x == 41) d[a] = -1e-30f;
               if (x == 42) d[a] = 1e25f;
               if (q % 16 == 1 && x == 43) d[a] = INFINITY;
               if (q % 16 == 1 && x == 44) d[a] = NAN;
               if (q % 16 == 1 && x == 45) o[a] = 1e20f;
               if (q % 16 == 1 && x == 46) o[a] = NAN;
               if (q % 16 == 1 && x == 47) o[a] = -INFINITY;
               if (x == 48) o[a] *= 1e5f;
            }
         }
         Ray r;
         make_ray(r, o[0], o[1], o[2], d[0], d[1], d[2]);
         const Seen want = binary(bvh, img, r);
         wide_ray(r);
         Seen got;
         uint32_t deepest = 0;
         rays++;
         if (!wide(w, img, r, got, deepest)) {
            handed++;
            continue;
         }
         hits += want.hit != 0xFFFFFFFFu;
         if (!got.same(want) || deepest > w.stack) {
            if (bad++ < 5)
               std::printf("scene %d ray %d: o %a %a %a d %a %a %a: %zu faces, want %zu; hit %u, want %u; stack %u of %u\n",
                           scene, q, o[0], o[1], o[2], d[0], d[1], d[2], got.faces.size(), want.faces.size(), got.hit,
                           want.hit, deepest, w.stack);
         }
      }
   }
   std::printf("%ld rays, %ld hits, %ld over the binary records, %ld mismatches\n", rays, hits, handed, bad);
   return bad || handed > rays / 20 || hits < rays / 20 ? 1 : 0;
}
