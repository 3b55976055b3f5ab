// Host check of the four-wide traversal of rays with direction components of
// -0 that start in the planes of flat leaves, over sheets, boxes and grids: the
// leaves, their order and the hit are those of the reference's traversal, and
// only rays without a bounded axis are left to the binary records.  Prints the
// numbers of rays and mismatches; exit 1 on a mismatch.
#include <hip/hip_runtime.h>

#include "wide.h"
#include "wide_build.h"

namespace {
// What the traversal makes of a passing leaf of `count` faces that is flat
// under -0 in `axes`: true when the ray is to be traced again; no faces when
// the reference does not reach the leaf.
bool flat_leaf(const ptx::WideImage &w, uint32_t axes, const ptx::dev::Ray &r, uint32_t first, uint32_t &count) {
   if (!axes) return false;
   if (r.nk & ptx::dev::kRayLoose) return true;
   if (axes & ~(first < w.flat.size() ? w.flat[first] : 0u)) count = 0;
   return false;
}
}  // namespace
#define wide_flat(a, b, c, d, e, f, r) flat_leaf(w, (wide_flat)(a, b, c, d, e, f, r), r, first, count)
#define main wide_check_main
#include "wide_check.cpp"
#undef main

int main() {
   std::mt19937 rng(37);
   auto uni = [&](float a, float b) { return a + (b - a) * float(rng() >> 8) * 0x1p-24f; };
   long rays = 0, bad = 0, handed = 0, loose = 0, hits = 0, flat = 0;
   for (int scene = 0; scene < 20; scene++) {
      // a sheet's two triangles a cell in one of the axes; boxes of six flat
      // sides on a grid; random sheets; faces with every corner on a small grid
      const int kind = scene % 4, axis = scene % 3;
      WorldMesh m;
      auto tri = [&](const float (&p)[3][3]) {
         for (auto &c : p)
            for (float x : c) m.wv.push_back(x);
         m.nf++;
      };
      auto quad = [&](int a, float at, float u0, float u1, float v0, float v1) {
         float c[4][3];
         for (int k = 0; k < 4; k++) {
            c[k][a] = at;
            c[k][(a + 1) % 3] = k & 1 ? u1 : u0;
            c[k][(a + 2) % 3] = k & 2 ? v1 : v0;
         }
         const float t0[3][3] = {{c[0][0], c[0][1], c[0][2]}, {c[1][0], c[1][1], c[1][2]}, {c[2][0], c[2][1], c[2][2]}};
         const float t1[3][3] = {{c[1][0], c[1][1], c[1][2]}, {c[3][0], c[3][1], c[3][2]}, {c[2][0], c[2][1], c[2][2]}};
         tri(t0);
         tri(t1);
      };
      if (kind == 0)
         for (int i = -3; i < 3; i++)
            for (int j = -3; j < 3; j++) quad(axis, 0.f, float(i), float(i + 1), float(j), float(j + 1));
      if (kind == 1)
         for (int n = 0; n < 12; n++) {
            const float o[3] = {float(int(rng() % 9) - 4), float(int(rng() % 9) - 4), float(int(rng() % 9) - 4)};
            for (int a = 0; a < 3; a++)
               for (int side = 0; side < 2; side++)
                  quad(a, o[a] + side, o[(a + 1) % 3], o[(a + 1) % 3] + 1, o[(a + 2) % 3], o[(a + 2) % 3] + 1);
         }
      if (kind == 2)
         for (int n = 0; n < 60; n++) {
            const float u = uni(-4, 3), v = uni(-4, 3);
            quad(int(rng() % 3), float(int(rng() % 5) - 2), u, u + uni(0, 1), v, v + uni(0, 1));
         }
      if (kind == 3)
         for (int n = 0; n < 80; n++) {
            float t[3][3];
            for (auto &c : t)
               for (float &x : c) x = float(int(rng() % 5) - 2);
            tri(t);
         }
      std::vector<WorldMesh> meshes = {m};
      HostBvh bvh;
      build_reference_bvh(meshes, 2, bvh);
      HostImage img;
      WideImage w;
      if (layout_scene(meshes, bvh, img) != PTX_OK || !build_wide(bvh, img, 2, w)) return 1;
      for (const uint8_t f : w.flat) flat += f != 0;
      for (int q = 0; q < 20000; q++) {
         const float odd[] = {0.f, -0.f, INFINITY, NAN, 1e-30f, 1e30f};
         float o[3], d[3];
         for (int a = 0; a < 3; a++) {
            o[a] = rng() % 4 ? float(int(rng() % 9) - 4) : uni(-5, 5);
            d[a] = rng() % 2 ? -0.f : q % 5 ? uni(-1, 1) : odd[rng() % 6];
            if (q % 50 == 0) o[a] = rng() % 2 ? -0.f : m.wv[rng() % m.wv.size()];
         }
         Ray r;
         make_ray(r, o[0], o[1], o[2], d[0], d[1], d[2]);
         const Seen want = binary(bvh, img, r);
         wide_ray(r);
         loose += (r.nk & kRayLoose) != 0;
         const bool may = (r.nk & kRayLoose) != 0;
         r.nk &= ~kRayHard;                        // wide_check.cpp's walk leaves such rays out
         Seen got;
         uint32_t deepest = 0;
         rays++;
         if (!wide(w, img, r, got, deepest)) {
            handed++;
            if (!may) bad++;
            continue;
         }
         hits += want.hit != 0xFFFFFFFFu;
         if (want.t != want.t && got.t != got.t) got.t = want.t;
         if (!got.same(want) || deepest > w.stack) {
            if (bad++ < 5)
               std::printf("scene %d ray %d: o %a %a %a d %a %a %a: %zu faces, want %zu; hit %u, want %u\n", scene, q,
                           o[0], o[1], o[2], d[0], d[1], d[2], got.faces.size(), want.faces.size(), got.hit, want.hit);
         }
      }
   }
   std::printf("%ld rays, %ld hits, %ld without a bounded axis, %ld traced again, %ld faces of flat leaves inside, "
               "%ld mismatches\n", rays, hits, loose, handed, flat, bad);
   return bad || hits < rays / 20 || flat == 0 ? 1 : 0;
}
