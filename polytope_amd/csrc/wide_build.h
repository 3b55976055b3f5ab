// Host builder of a scene's four-wide form (wide_build.cpp); its face records
// are made on the device (launch_build_wide_faces).
#pragma once

#include "scene.h"

namespace ptx {

struct WideImage {
   UnsetVector<WideNode> nodes;
   std::vector<WideLeaf> leaves;    // leaf 0 is empty
   UnsetVector<uint8_t> flat;       // WideFace::flat of every face, or nothing where no leaf is flat
   uint32_t root = 0;               // wide node or leaf reference
   uint32_t stack = 1;              // 8-byte stack entries a lane needs
};

// False, with `out` unspecified, when the tree has no wide form: boxes that do
// not nest, or are not finite, or indices past what its references hold.
// threads 0 = all host cores.
bool build_wide(const HostBvh &bvh, const HostImage &img, unsigned threads, WideImage &out);

}  // namespace ptx
