// Internal declarations shared by the host C++ and HIP translation units of
// libptx_hip.so.  Not part of the C ABI (include/ptx.h).
#pragma once

#include <cstddef>
#include <cstdint>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "../../include/ptx.h"

namespace ptx {

// ---------------------------------------------------------------- device layout
//
// Interior node record, 64 bytes, one per interior node of the reference BVH in
// DFS order.  Child 0 is the reference's low child (node i+1), child 1 its high
// child (node i + high_child_offset).  A child reference with bit 31 set is a
// leaf and holds the index of its first triangle in the leaf-ordered triangle
// array (the reference's leaf_ordered_indices order); the leaf's face count (the
// reference's u16 num_faces) sits in `counts`.  Otherwise the reference is the
// index of the child's interior record.
//   f[0..5]   child 0 box p0.xyz, p1.xyz
//   f[6..11]  child 1 box p0.xyz, p1.xyz
//   u[12]     child 0 ref, u[13] child 1 ref
//   u[14]     child 0 slot | child 1 slot << 16: a leaf child's face count,
//             an interior child's split axis
//   u[15]     split axis
struct alignas(64) Node64 {
   float box[12];
   uint32_t ref[2];
   uint32_t counts;
   uint32_t axis;
};
static_assert(sizeof(Node64) == 64, "Node64 is 64 bytes");

constexpr uint32_t kLeafBit = 0x80000000u;

// Four-wide form of the tree (wide.h): up to four descendants of a binary
// node, their boxes in steps of 2^(exponent - 24) from the node's low corner,
// rounded outwards (a plane's byte read as a half is 2^-24 times its steps).  planes: low and high x, low and high y, low and high z, child k in
// byte k.  later[q], q = octant of the rays whose z direction is not negative
// (bit a set: direction a negative): bits 4 k .. 4 k + 3 = the children visited
// after child k; the octant with every sign flipped visits in reverse.  Only
// the children in `used` (bit k) are there: an empty one (low 255, high 0) may
// pass a test and has no place in the order.
struct alignas(64) WideNode {
   float org[3];
   int8_t exponent[3];       // x, y, z
   uint8_t used;
   uint8_t planes[6][4];
   uint32_t ref[4];
   uint16_t later[4];
};
static_assert(sizeof(WideNode) == 64, "WideNode is 64 bytes");

// A face as the four-wide traversal reads it, at its leaf-ordered index.  flat,
// of a leaf's first face: the axes (bit a) in which the leaf's box is flat and
// the smallest box above it that is not holds its coordinate strictly inside.
struct alignas(16) WideFace {
   float v[9];               // world v0, v1, v2
   uint32_t mesh, face;      // the reference's ids
   uint32_t flat;
};
static_assert(sizeof(WideFace) == 48, "WideFace layout");

// A leaf of more than two faces, or whose box is not its corners': leaf 0 of a
// scene is the empty one.
struct alignas(16) WideLeaf {
   float box[6];
   uint32_t first, count;
};
static_assert(sizeof(WideLeaf) == 32, "WideLeaf layout");

// Per-mesh shading record (9 words, read as one block by the shading step).
// Glossy meshes that are not lights keep the lobe's constant reflectance in
// refl and its roughness in emission[0].  A textured Lambert mesh
// (kRecTextured) takes its reflectance from its triangles' texture records.
constexpr uint32_t kRecNormals = 1u, kRecTextured = 2u;
struct MeshRec {
   int32_t brdf;
   float refl[3];
   int32_t is_light;
   float emission[3];
   uint32_t flags;           // kRecNormals | kRecTextured
};
static_assert(sizeof(MeshRec) == 36, "MeshRec layout");

// Texture record of one leaf-ordered triangle (32 bytes), present for every
// triangle of a scene with textured meshes: its corner texture coordinates,
// the texture's size and whether the triangle is textured, and the offset of
// the texture's first texel in the scene's texel pool, which follows the
// num_tris records in the same allocation.
constexpr uint32_t kTexTextured = 1u << 31, kTexNormals = 1u << 30;
struct TexTri {
   float uv[6];              // (u, v) of corners 0, 1, 2 (fv0, fv1, fv2)
   uint32_t wh;              // width | height << 15 | kTexNormals | kTexTextured
   uint32_t texel0;          // first texel of the texture in the pool
};
static_assert(sizeof(TexTri) == 32, "TexTri layout");

// Device view of one scene.  The first 48 bytes are what a traversal needs
// (loaded per lane by the render path's extend stage as three 16-byte loads).
struct DevScene {
   const Node64 *nodes;      // interior records
   const float *tris;        // 9 floats (world v0, v1, v2) per leaf-ordered triangle
   float root_box[6];
   uint32_t root_ref;        // kLeafBit|first triangle, or interior index
   uint32_t root_count;      // face count when the root is a leaf
   const uint32_t *pairs;    // (mesh, face) per leaf-ordered triangle
   const MeshRec *meshes;
   const float *normals;     // world corner normals, 9 floats per leaf-ordered triangle (or null)
   uint32_t num_tris;
   uint32_t max_stack;       // deepest deferred-stack use + 1 (tree depth bound)
   float sky[3];
   uint16_t num_lights;
   uint16_t has_sky;
   const float *lights;      // point lights, 6 floats each (position, intensity), or null
   const TexTri *tex_tris;   // texture records per leaf-ordered triangle, then the texel pool; or null
};
static_assert(sizeof(DevScene) == 112, "DevScene layout");

// Device view of a scene's four-wide form.
struct WideScene {
   const WideNode *nodes;
   const WideFace *faces;    // null: the scene has no such form
   const WideLeaf *leaves;
   uint32_t root;            // a node's index or a leaf reference
   uint32_t stack;           // 8-byte stack entries a lane needs, the sentinel and exact_trace's words among them
};

// Per-job constants of a render, device-resident in the job table.
struct JobDev {
   float cam[16];            // camera-to-world, row-major
   float oow, ooh, aspect, tanf2;
   uint32_t width, height, spp, max_depth;
   uint32_t seed, scene;     // RNG seed; index into the scene table
   uint32_t flags, pad;      // PTX_JOB_*
   float *film;              // W*H*3 running sums (BoxFilter order), then the average
   uint32_t *primary;        // W*H primary-hit records (16 words each)
};

// A contiguous block of path slots: samples [s0, s0 + k) of every pixel of a job.
// Slot of (pixel p, sample s) = base + (s - s0) * npix + p.
struct Chunk {
   uint32_t job, s0, k, npix, base;
};

// How a persistent launch's ids are dealt out: `batches` batches of `batch`
// consecutive ids, the first static_batches of them round robin to the waves,
// the rest by a counter.
struct Deal {
   uint32_t n, batch, batches, static_batches;
};

// Largest number of chunks in a round of the path-regeneration kernel (its
// chunk table lives in LDS).
constexpr uint32_t kMaxRoundChunks = 64;

// ---------------------------------------------------------------- host-side scene

// A vector whose resize leaves new elements unset: large arrays that several
// threads fill are then first touched by those threads.
template <class T>
struct UnsetAlloc : std::allocator<T> {
   template <class U>
   struct rebind {
      using other = UnsetAlloc<U>;
   };
   template <class U, class... A>
   void construct(U *p, A &&...a) {
      if constexpr (sizeof...(A) == 0) ::new (static_cast<void *>(p)) U;
      else ::new (static_cast<void *>(p)) U(std::forward<A>(a)...);
   }
};
template <class T>
using UnsetVector = std::vector<T, UnsetAlloc<T>>;

struct HostBvh {
   std::vector<ptx_bvh_node> nodes;       // reference compact layout
   std::vector<uint32_t> pairs;           // 2 per leaf entry (mesh, face)
};

struct WorldMesh {
   uint32_t nf = 0;
   UnsetVector<float> wv;                 // 9 floats per face (world v0, v1, v2)
   bool has_normals = false;
   UnsetVector<float> wn;                 // 9 floats per face (world corner normals)
   std::vector<float> uv;                 // textured: 6 floats per face (u, v of corners 0, 1, 2)
   int32_t texture = -1;                  // textured: index into the scene's texture table
   MeshRec rec{};
};

// Transform::ApplyInPlace(Point&) semantics (src/cpu/structures/Transform.cpp:69-91).
// shading: also the mesh record and a textured mesh's corner coordinates (whose
// indices the caller has checked against num_uv).
void world_vertices(const ptx_mesh_desc &m, WorldMesh &out, bool shading = true);

// Decision-identical re-implementation of bvh::bound + bvh::compact
// (src/cpu/acceleration/bvh.cpp:36-395, 652-698), multithreaded.
void build_reference_bvh(const std::vector<WorldMesh> &meshes, unsigned threads, HostBvh &out);

// Error reporting: per-thread message returned by ptx_last_error().
int set_error(int code, const std::string &msg);

}  // namespace ptx
