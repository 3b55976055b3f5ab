// Host check of ptx_render at memory limits: wherever one launch per sample
// finds its memory the default form renders too, on a fresh device and behind a
// job that left its path slots, and closing the device leaves nothing.  Prints
// the failures; exit 1 on any.
#include <cstdio>

#include "host_runtime.h"
#include "ptx.h"

static ptx_job_desc job_of(uint32_t side, uint32_t spp, bool nee) {
   ptx_job_desc j{};
   for (int k = 0; k < 4; k++) j.camera.camera_to_world[5 * k] = 1.f;
   j.camera.width = j.camera.height = side;
   j.camera.one_over_width = j.camera.one_over_height = 1.f / float(side);
   j.camera.aspect_ratio = j.camera.tan_fov_over_2 = 1.f;
   j.spp = spp;
   j.max_depth = 5;
   j.flags = nee ? PTX_JOB_NEE : 0u;
   return j;
}

// One device with a scene of a triangle and a light; renders `first` (spp > 0)
// and then `job`, the limit set once the scene is there.
static int render(size_t limit, uint32_t form, const ptx_job_desc &first, const ptx_job_desc &job, size_t &left) {
   host_runtime::State &rt = host_runtime::state();
   rt.limit = SIZE_MAX;
   const size_t base = rt.used;
   ptx_device *dev = nullptr;
   if (ptx_device_open(0, &dev) != PTX_OK) return -1;
   const float x[3] = {0, 1, 0}, y[3] = {0, 0, 1}, z[3] = {2, 2, 2};
   const uint32_t f[3] = {0, 1, 2};
   ptx_mesh_desc m{};
   m.num_vertices = 3;
   m.num_faces = 1;
   m.x = x; m.y = y; m.z = z;
   m.fv0 = f; m.fv1 = f + 1; m.fv2 = f + 2;
   m.brdf = PTX_BRDF_LAMBERT;
   for (int k = 0; k < 4; k++) m.object_to_world[5 * k] = m.world_to_object[5 * k] = 1.f;
   ptx_point_light light{};
   ptx_scene_desc desc{};
   desc.meshes = &m;
   desc.num_meshes = 1;
   desc.lights = &light;
   desc.num_lights = 1;
   ptx_scene *scene = nullptr;
   if (ptx_scene_create(dev, &desc, &scene) != PTX_OK) return -1;
   ptx_tuning t{};
   t.plain_primary = form;
   (void)ptx_set_tuning(dev, &t);
   std::vector<float> film(3 * 512 * 512);
   int rc = PTX_OK;
   if (first.spp) rc = ptx_render(scene, &first, film.data());
   rt.limit = rt.used + limit;
   if (first.spp) rt.limit = base + limit;
   rc = ptx_render(scene, &job, film.data());
   rt.limit = SIZE_MAX;
   ptx_scene_destroy(scene);
   ptx_device_close(dev);
   left = rt.used - base;
   return rc;
}

int main() {
   int bad = 0;
   uint32_t both = 0, neither = 0;
   for (const bool nee : {false, true})
      for (const bool behind : {false, true}) {
         // 256 x 256 pixels and 64 samples: 5 MB of film and primary records, 50 MB of path slots; with next-event
         // estimation one sample behind a job that left 30 MB
         const ptx_job_desc job = nee && behind ? job_of(512, 1, nee) : job_of(256, 64, nee);
         const ptx_job_desc first = behind ? job_of(200, 64, false) : ptx_job_desc{};
         for (size_t limit = 0; limit < (size_t(96) << 20); limit += 769 << 10) {
            size_t left[2] = {0, 0};
            const int launches = render(limit, PTX_PLAIN_CACHED, first, job, left[0]);
            const int rc = render(limit, PTX_PLAIN_DEFAULT, first, job, left[1]);
            if (launches == PTX_OK && rc != PTX_OK)
               std::printf("limit %zu nee %d behind %d: %s\n", limit, nee, behind, ptx_last_error()), bad++;
            if (left[0] || left[1]) std::printf("limit %zu: %zu and %zu bytes left\n", limit, left[0], left[1]), bad++;
            if (launches == PTX_OK) both++;
            else neither++;
         }
      }
   std::printf("%u limits with memory, %u without, %d failures\n", both, neither, bad);
   return bad || !both || !neither;
}
