// Host check of the four-wide traversal of rays whose components are not
// finite or whose direction is zero, over the scenes of wide_check.cpp: none
// starts over the binary records, and the leaves, their order and the hit are
// those of the reference's traversal.  Such rays come in numbers: a program
// marks the idle lanes of a batch with them.  Prints the numbers of rays and
// mismatches; exit 1 on a mismatch.
#define main wide_check_main
#include "wide_check.cpp"
#undef main

int main() {
   std::mt19937 rng(29);
   auto uni = [&](float a, float b) { return a + (b - a) * float(rng() >> 8) * 0x1p-24f; };
   long rays = 0, bad = 0, handed = 0, hits = 0, nan_hits = 0, exact = 0;
   for (int scene = 0; scene < 12; scene++) {
      // random faces, faces on an integer grid, flat sheets, one to three faces
      const int kind = scene % 4;
      const uint32_t nf = kind == 3 ? 1 + scene / 4 : 50u << (scene / 2);
      WorldMesh m;
      m.nf = nf;
      m.wv.resize(9 * size_t(nf));
      for (uint32_t f = 0; f < nf; f++) {
         const float c[3] = {uni(-4, 4), uni(-4, 4), uni(-4, 4)};
         for (int v = 0; v < 3; v++)
            for (int a = 0; a < 3; a++) {
               float x = c[a] + uni(-0.6f, 0.6f);
               if (kind == 1) x = std::round(x);
               if (kind == 2 && a == (int)(f % 3)) x = float(int(f % 5) - 2);
               m.wv[9 * size_t(f) + 3 * v + a] = x;
            }
      }
      std::vector<WorldMesh> meshes = {m};
      HostBvh bvh;
      build_reference_bvh(meshes, 2, bvh);
      HostImage img;
      WideImage w;
      if (layout_scene(meshes, bvh, img) != PTX_OK || !build_wide(bvh, img, 2, w)) return 1;
      for (int q = 0; q < 20000; q++) {
         const float odd[] = {0.f, -0.f, INFINITY, -INFINITY, NAN, 1e38f, -1e-39f, 1.f};
         float o[3], d[3];
         for (int a = 0; a < 3; a++) {
            o[a] = uni(-6, 6);
            if (q % 3) o[a] = std::round(o[a]);
            d[a] = q % 8 == 0 ? rng() % 2 ? 0.f : -0.f : uni(-1, 1);
            if (q % 8 > 1 && rng() % 3 == 0) d[a] = odd[rng() % 8];
            if (q % 8 > 4 && rng() % 4 == 0) o[a] = odd[rng() % 8];
         }
         Ray r;
         make_ray(r, o[0], o[1], o[2], d[0], d[1], d[2]);
         const Seen want = binary(bvh, img, r);
         wide_ray(r);
         Trav t;
         t.r = r;
         wide_begin(t, img.root_box, w.root);
         exact += t.cur == kWideExact;
         r.nk &= ~kRayHard;                        // wide_check.cpp's walk leaves such rays out
         Seen got;
         uint32_t deepest = 0;
         rays++;
         if (!wide(w, img, r, got, deepest)) {     // flat at the origin under -0
            handed++;
            continue;
         }
         hits += want.hit != 0xFFFFFFFFu;
         nan_hits += want.t != want.t;
         // NaN distances of either sign and payload are one: the two walks are compiled apart
         if (want.t != want.t && got.t != got.t) got.t = want.t;
         if (!got.same(want) || deepest > w.stack) {
            if (bad++ < 5)
               std::printf("scene %d ray %d: o %a %a %a d %a %a %a: %zu faces, want %zu; hit %u, want %u\n", scene, q,
                           o[0], o[1], o[2], d[0], d[1], d[2], got.faces.size(), want.faces.size(), got.hit, want.hit);
         }
      }
   }
   std::printf("%ld rays, %ld hits, %ld of them at NaN, %ld traced again, %ld started over the binary records, "
               "%ld mismatches\n", rays, hits, nan_hits, handed, exact, bad);
   return bad || exact || handed > rays / 10 || hits < rays / 20 || nan_hits < rays / 100 ? 1 : 0;
}
