// Host check of ptx_scene_create at every memory limit: a scene with corner
// normals, a texture and a light is created wherever the arrays that it cannot
// do without fit, with its four-wide form only where that fits too, and no
// limit leaves an allocation behind.  A creation makes two allocations and, of
// a small scene, two copies and no launch.  Prints the failures; exit 1 on any.
#include <cmath>
#include <cstdio>

#include "host_runtime.h"
#include "ptx.h"

// A sheet of 2 side^2 faces; returns the number of failures.  A form of 16 MB
// or more (large) is made only where it leaves an eighth of the memory.
static int check(uint32_t kSide, bool large, uint32_t steps) {
   const uint32_t kVerts = (kSide + 1) * (kSide + 1), kFaces = 2 * kSide * kSide, kTex = 16;
   std::vector<float> x(kVerts), y(kVerts), z(kVerts), up(kVerts, 1.f), flat(kVerts, 0.f), u(kVerts), v(kVerts);
   for (uint32_t i = 0; i < kVerts; i++) {
      x[i] = float(i % (kSide + 1));
      z[i] = float(i / (kSide + 1));
      y[i] = std::sin(x[i]) * std::cos(z[i]);
      u[i] = x[i] / kSide;
      v[i] = z[i] / kSide;
   }
   std::vector<uint32_t> f0, f1, f2;
   for (uint32_t i = 0; i < kSide; i++)
      for (uint32_t j = 0; j < kSide; j++) {
         const uint32_t a = i * (kSide + 1) + j, b = a + 1, c = a + kSide + 1, d = c + 1;
         f0.push_back(a); f1.push_back(b); f2.push_back(c);
         f0.push_back(b); f1.push_back(d); f2.push_back(c);
      }
   std::vector<uint8_t> texels(4 * kTex * kTex, 100);
   ptx_texture_desc tex{};
   tex.rgba = texels.data();
   tex.width = tex.height = kTex;
   ptx_point_light light{};
   ptx_mesh_desc m{};
   m.num_vertices = m.num_uv = kVerts;
   m.num_faces = kFaces;
   m.x = x.data(); m.y = y.data(); m.z = z.data();
   m.nx = flat.data(); m.ny = up.data(); m.nz = flat.data();
   m.fv0 = f0.data(); m.fv1 = f1.data(); m.fv2 = f2.data();
   m.u = u.data(); m.v = v.data();
   m.brdf = PTX_BRDF_LAMBERT;
   m.texture = 1;
   for (int k = 0; k < 4; k++) m.object_to_world[5 * k] = m.world_to_object[5 * k] = 1.f;
   ptx_scene_desc desc{};
   desc.meshes = &m;
   desc.num_meshes = 1;
   desc.textures = &tex;
   desc.num_textures = 1;
   desc.lights = &light;
   desc.num_lights = 1;
   host_runtime::State &rt = host_runtime::state();
   ptx_device *dev = nullptr;
   if (ptx_device_open(0, &dev) != PTX_OK) return std::printf("no device: %s\n", ptx_last_error()), 1;
   const size_t base = rt.used;
   ptx_scene *scene = nullptr;
   ptx_scene_info info{};
   const uint32_t allocations = rt.allocations, copies = rt.copies;
   const size_t launches = rt.launches.size();
   if (ptx_scene_create(dev, &desc, &scene) != PTX_OK) return std::printf("no scene: %s\n", ptx_last_error()), 1;
   int bad = 0;
   const uint32_t a = rt.allocations - allocations, c = rt.copies - copies, l = uint32_t(rt.launches.size() - launches);
   if (a != 2 || (kFaces <= 1152 ? c != 2 || l != 0 : l != 1))
      std::printf("%u faces: %u allocations, %u copies, %u launches\n", kFaces, a, c, l), bad++;
   (void)ptx_scene_get_info(scene, &info);
   const size_t whole = rt.used - base;
   // records, triangles with their padding, ids, mesh record, texture records and texels, corner normals,
   // light; seven arrays, which may be padded to 256 bytes each
   const size_t least = size_t(info.num_interior) * 64 + size_t(kFaces) * 36 + 128 + size_t(info.num_pairs) * 8 + 36 +
                        size_t(kFaces) * 32 + 4 * kTex * kTex + size_t(kFaces) * 36 + 24;
   if (info.device_bytes != whole) std::printf("%zu bytes used, %zu told\n", whole, (size_t)info.device_bytes), bad++;
   ptx_scene_destroy(scene);
   // what it takes without the form: at the largest limit that the whole misses
   rt.limit = base + whole - (large ? 0 : 1);
   if (ptx_scene_create(dev, &desc, &scene) != PTX_OK) return std::printf("refused: %s\n", ptx_last_error()), 1;
   const size_t need = rt.used - base;
   if (need < least || need > least + 7 * 256) std::printf("%zu bytes without the form, %zu needed\n", need, least), bad++;
   ptx_scene_destroy(scene);
   uint32_t with = 0, without = 0, refused = 0;
   const size_t most = large ? whole * 5 / 4 : whole, step = most / steps + 1;
   for (size_t limit = 0; limit <= most; limit += limit + step < most ? step : std::max<size_t>(1, most - limit)) {
      rt.limit = base + limit;
      scene = nullptr;
      const int rc = ptx_scene_create(dev, &desc, &scene);
      const size_t used = rt.used - base;
      if (rc == PTX_OK) {
         (void)ptx_scene_get_info(scene, &info);
         if (limit < need || used != info.device_bytes || used != (limit < whole || (large && limit - whole < (base + limit) / 8) ? need : whole))
            std::printf("limit %zu: a scene of %zu bytes, %zu told\n", limit, used, (size_t)info.device_bytes), bad++;
         (used == whole ? with : without)++;
         ptx_scene_destroy(scene);
      } else {
         if (limit >= need) std::printf("limit %zu: refused, %zu needed: %s\n", limit, need, ptx_last_error()), bad++;
         refused++;
      }
      if (rt.used != base) std::printf("limit %zu: %zu bytes left\n", limit, rt.used - base), bad++;
      if (hipGetLastError() != hipSuccess) std::printf("limit %zu: an error left for the caller\n", limit), bad++;
      if (limit == most) break;
   }
   rt.limit = SIZE_MAX;
   ptx_device_close(dev);
   std::printf("%u scenes with the four-wide form, %u without, %u refused\n", with, without, refused);
   return bad + (!with || !without || !refused);
}

int main() {
   int bad = 0;
   for (uint32_t side : {4u, 24u, 48u}) bad += check(side, false, 211);      // 32, 1,152 and 4,608 faces
   bad += check(400, true, 17);                                              // 320,000
   std::printf("%d failures\n", bad);
   return bad != 0;
}
