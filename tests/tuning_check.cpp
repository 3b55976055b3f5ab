// Host check of ptx_get_tuning: the fields whose default depends on the form a
// kernel steps over come back as they were set, so that setting back what was
// got, or that with one field changed, changes no other.  Prints the failures;
// exit 1 on any.
#include <cstdio>

#include "host_runtime.h"
#include "ptx.h"

int main() {
   ptx_device *dev = nullptr;
   if (ptx_device_open(0, &dev) != PTX_OK) return 1;
   int bad = 0;
   ptx_tuning t{}, back{};
   (void)ptx_get_tuning(dev, &t);
   if (t.refill_lanes || t.shade_lanes || t.leaf_lanes || t.blocks_per_cu || t.paths_per_wave)
      std::printf("unset: refill %u shade %u leaf %u\n", t.refill_lanes, t.shade_lanes, t.leaf_lanes), bad++;
   if (t.lds_stack != 12 || t.block_size != 256) std::printf("unset: lds %u block %u\n", t.lds_stack, t.block_size), bad++;
   for (uint32_t refill : {0u, 4u, 16u})
      for (uint32_t shade : {0u, 16u, 48u}) {
         t.refill_lanes = refill;
         t.shade_lanes = shade;
         (void)ptx_set_tuning(dev, &t);
         (void)ptx_get_tuning(dev, &back);
         if (std::memcmp(&t, &back, sizeof t)) std::printf("refill %u shade %u came back as %u %u\n", refill, shade,
                                                           back.refill_lanes, back.shade_lanes), bad++;
      }
   ptx_device_close(dev);
   std::printf("%d failures\n", bad);
   return bad != 0;
}
