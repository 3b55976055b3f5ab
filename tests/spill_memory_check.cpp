// Host check of the stack spill at memory limits: wherever a scene without a
// four-wide form renders (a batch, with next-event estimation, over wavefront
// queues, one launch per sample) or answers device rays, the same scene with
// one does too, although its stack asks for more.  Prints the failures; exit 1
// on any.
#include <cmath>
#include <cstdio>

#include "host_runtime.h"
#include "ptx.h"

enum Call { kBatch, kBatchNee, kWavefront, kLaunches, kRays, kCalls };

static ptx_job_desc job_of(uint32_t w, uint32_t h, uint32_t spp, bool nee) {
   ptx_job_desc j{};
   for (int k = 0; k < 4; k++) j.camera.camera_to_world[5 * k] = 1.f;
   j.camera.width = w;
   j.camera.height = h;
   j.camera.one_over_width = 1.f / float(w);
   j.camera.one_over_height = 1.f / float(h);
   j.camera.aspect_ratio = j.camera.tan_fov_over_2 = 1.f;
   j.spp = spp;
   j.max_depth = 5;
   j.flags = nee ? PTX_JOB_NEE : 0u;
   return j;
}

// A sheet of 40 x 40 triangles.
static int make_scene(ptx_device *dev, ptx_scene **scene) {
   const uint32_t side = 40, n = side * side;
   std::vector<float> x, y, z;
   std::vector<uint32_t> f[3];
   for (uint32_t i = 0; i < n; i++)
      for (uint32_t k = 0; k < 3; k++) {
         const uint32_t u = i % side, v = i / side;
         x.push_back(float(u + (k == 1)));
         y.push_back(std::sin(float(u * v)));
         z.push_back(float(v + (k == 2)));
         f[k].push_back(3 * i + k);
      }
   ptx_mesh_desc m{};
   m.num_vertices = 3 * n;
   m.num_faces = n;
   m.x = x.data(); m.y = y.data(); m.z = z.data();
   m.fv0 = f[0].data(); m.fv1 = f[1].data(); m.fv2 = f[2].data();
   m.brdf = PTX_BRDF_LAMBERT;
   for (int k = 0; k < 4; k++) m.object_to_world[5 * k] = m.world_to_object[5 * k] = 1.f;
   ptx_point_light light{};
   ptx_scene_desc desc{};
   desc.meshes = &m;
   desc.num_meshes = 1;
   desc.lights = &light;
   desc.num_lights = 1;
   desc.build_threads = 1;
   return ptx_scene_create(dev, &desc, scene);
}

// The call's result with `limit` bytes over the scene's; wide: a scene with the
// form, which is made last and left out where its memory is missing.
static int run(Call call, size_t limit, bool wide) {
   host_runtime::State &rt = host_runtime::state();
   rt.limit = SIZE_MAX;
   ptx_device *dev = nullptr;
   ptx_scene *scene = nullptr;
   if (ptx_device_open(0, &dev) != PTX_OK || make_scene(dev, &scene) != PTX_OK) return -1;
   if (!wide) {
      const size_t all = rt.used;
      ptx_scene_destroy(scene);
      rt.limit = all - 1;
      if (make_scene(dev, &scene) != PTX_OK || rt.used >= all) return -1;
   }
   rt.limit = rt.used + limit;
   static std::vector<float> film[2] = {std::vector<float>(3 * 512 * 400), std::vector<float>(3 * 256 * 256)};
   int rc = -1;
   if (call == kRays) {
      float rays[6] = {0};
      ptx_hit hit;
      rc = ptx_intersect_closest_device(scene, rays, 1 << 20, &hit, nullptr, nullptr, nullptr);
   } else {
      const bool nee = call == kBatchNee;
      ptx_tuning t{};
      if (call == kWavefront) {
         t.render_mode = PTX_RENDER_WAVEFRONT;
         t.paths_per_wave = 1 << 18;
      } else if (call == kLaunches) {
         t.plain_primary = PTX_PLAIN_RETRACE;
      }
      (void)ptx_set_tuning(dev, &t);
      const ptx_job_desc jobs[2] = {job_of(512, 400, 4, nee), job_of(256, 256, 16, nee)};
      ptx_scene *scenes[2] = {scene, scene};
      float *films[2] = {film[0].data(), film[1].data()};
      rc = call == kLaunches ? ptx_render(scene, jobs, films[0]) : ptx_render_batch(scenes, jobs, 2, films);
   }
   rt.limit = SIZE_MAX;
   ptx_scene_destroy(scene);
   ptx_device_close(dev);
   return rc;
}

int main() {
   int bad = 0;
   uint32_t both = 0, neither = 0;
   for (int call = 0; call < kCalls; call++)
      for (size_t limit = 0; limit < (size_t(110) << 20); limit += 1511 << 10) {
         const int plain = run(Call(call), limit, false), rc = run(Call(call), limit, true);
         if (plain == PTX_OK && rc != PTX_OK)
            std::printf("call %d limit %zu: %s\n", call, limit, ptx_last_error()), bad++;
         if (plain == PTX_OK) both++;
         else neither++;
      }
   std::printf("%u limits with memory, %u without, %d failures\n", both, neither, bad);
   return bad || !both || !neither;
}
