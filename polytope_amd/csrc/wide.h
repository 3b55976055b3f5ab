// Four-wide form of the reference tree: its layout, the conservative child
// test, and the traversal that visits the reference's leaves in the
// reference's order.
//
// Why the leaves are the same.  The reference visits a leaf when the leaf's
// box and every ancestor's box pass BoundingBox::Hits, each against the MinT
// of its own pop.  In a tree whose boxes nest, an ancestor's box passes
// whenever the leaf's does: every slab value is a monotone function of the
// plane in float arithmetic, so the ancestor's near is no larger and its far
// no smaller, and its pop came earlier, at a MinT no smaller.  So the leaves
// visited are exactly those whose own box passes at their turn, in the order
// the split-axis signs give, whatever skips the subtrees in between, as long
// as no skipped subtree holds a passing leaf.  A wide node therefore holds up
// to four descendants of a binary node with the visiting order of each
// direction octant, tests them conservatively (boxes in 8-bit steps, one fma a plane), and the
// leaf's exact box is tested when its turn comes.
//
// The one case in which boxes do not nest as tests: a direction component of
// -0 makes the reference's slab selections accept a box that is flat in that
// axis at the origin's coordinate c inside boxes they reject, those with c on
// their face.  Of the boxes above such a leaf those that are flat too pass, and
// of the others the smallest decides: c inside it is inside all of them, and c on
// its face is rejected there, its interval starting or ending at infinity.  So
// whether the leaf is visited is known beforehand (WideFace::flat), but for a
// ray whose other axes leave the interval's end at infinity (kRayLoose): that
// is traced again over the binary records in the reference's own steps
// (exact_trace).  Rays with NaN, infinite or all-zero components nest: a NaN
// slab value leaves the fold as it was in every box, and an infinite one moves
// with the plane as a finite one does.
#pragma once

#include "traverse.h"

#pragma clang fp contract(off)

namespace ptx {

// Child references: bit 31 clear = a wide node's index; set = a leaf, bits
// 29-30 its kind, bits 0-28 an index.
constexpr uint32_t kWideIndex = 0x1FFFFFFFu;
constexpr uint32_t kWideHeader = kLeafBit;                  // WideLeaf index: box and face range
constexpr uint32_t kWideOne = kLeafBit | (1u << 29);        // one face, whose corners span the leaf's box
constexpr uint32_t kWideTwo = kLeafBit | (2u << 29);        // two faces, likewise
constexpr uint32_t kWideRaw = kLeafBit | (3u << 29);        // Trav::cnt faces whose leaf's box has passed
constexpr uint32_t kWideExact = 0xFFFFFFFEu;                // trace again over the binary records

// Wide-test constants: the slack that covers the rounding of (corner - o) * i
// and of the added slack (3 units at most, 4 taken), and the factor that
// covers the relative rounding of the reference's slab values and of the fma
// against them, the reference's own far scale among it (13 units at most).
// The steps themselves add no error: a step times 1 / d is exact, and the
// builder rounds planes outwards in double.
constexpr float kWideSlack = 4 * 5.9604644775390625e-8f;
constexpr float kWideFar = 1 + 16 * 5.9604644775390625e-8f;
constexpr float kWideTiny = 0x1p-120f;     // covers underflow, whose error is absolute
// Rays whose |origin| or |1 / direction| reach this take the exact slab in
// place of the fma form, which could overflow (2^53.2 times a step of 2^47 in
// units of 2^24); scenes that reach it have no wide form.
constexpr float kWideLimit = 1e16f;
// A node's exponents are in units of 2^-24 steps: wide_step.
constexpr int kWideStep = 24;


namespace dev {

// Ray::nk bits beside the signs and the Wald axis
constexpr uint32_t kRayAxisShift = 3, kRayAxisMask = 3u;
constexpr uint32_t kRaySlow = 1u << 5;     // child tests with the exact slab
constexpr uint32_t kRayMinus = 1u << 6;    // some 1 / direction is -inf
constexpr uint32_t kRayHard = 1u << 7;     // an accepted face's t may be NaN: a component is not finite, or all are 0
constexpr uint32_t kRayLoose = 1u << 14;   // kRayMinus, and no axis bounds every box's interval
// 16 * the octant's entry of WideNode::later, in bits 8-13
constexpr uint32_t kRayLaterShift = 8;
constexpr uint32_t kLaterFlip = 0x7BDEu;   // every pair of different children

// Classifies a ray set up by make_ray (adds the kRay* bits to nk).
PTX_HD void wide_ray(Ray &r) {
   r.nk |= (((r.nk & 4u) ? ~r.nk : r.nk) & 3u) << (kRayLaterShift + 4);
   const float ax = __builtin_fabsf(r.ix), ay = __builtin_fabsf(r.iy), az = __builtin_fabsf(r.iz);
   const float mo = fmaxf(fmaxf(__builtin_fabsf(r.ox), __builtin_fabsf(r.oy)), __builtin_fabsf(r.oz));
   // fmaxf skips NaN: every component is compared by itself
   const bool plain = ax < kWideLimit && ay < kWideLimit && az < kWideLimit && mo < kWideLimit && r.ox == r.ox &&
                      r.oy == r.oy && r.oz == r.oz && ax > 0.f && ay > 0.f && az > 0.f;
   if (plain) return;
   uint32_t f = kRaySlow;
   if (r.ix == -kInf || r.iy == -kInf || r.iz == -kInf) {
      const bool bounded = (ax < kWideLimit && __builtin_fabsf(r.ox) < kWideLimit) ||
                           (ay < kWideLimit && __builtin_fabsf(r.oy) < kWideLimit) ||
                           (az < kWideLimit && __builtin_fabsf(r.oz) < kWideLimit);
      f |= bounded ? kRayMinus : kRayMinus | kRayLoose;
   }
   const bool nan = !(r.ix == r.ix && r.iy == r.iy && r.iz == r.iz && r.ox == r.ox && r.oy == r.oy && r.oz == r.oz);
   const bool all_inf = ax == kInf && ay == kInf && az == kInf;
   if (nan || all_inf || !(ax > 0.f && ay > 0.f && az > 0.f) || mo == kInf) f |= kRayHard;
   r.nk |= f;
}

// A node's frame for one ray: the entry of a plane at step q is q * s + l (a
// plane the ray enters through) or q * s + h (one it leaves through), with q in
// units of 2^-24 (wide_step) and s accordingly larger.
struct WideFrame {
   float sx, sy, sz, lx, ly, lz, hx, hy, hz;
};
PTX_HD WideFrame wide_frame(const Ray &r, float gx, float gy, float gz, int ex, int ey, int ez) {
   const float x = (gx - r.ox) * r.ix, y = (gy - r.oy) * r.iy, z = (gz - r.oz) * r.iz;
   WideFrame w;
   w.sx = __builtin_ldexpf(r.ix, ex);
   w.sy = __builtin_ldexpf(r.iy, ey);
   w.sz = __builtin_ldexpf(r.iz, ez);
   w.lx = __builtin_fmaf(__builtin_fabsf(x), -kWideSlack, x);
   w.ly = __builtin_fmaf(__builtin_fabsf(y), -kWideSlack, y);
   w.lz = __builtin_fmaf(__builtin_fabsf(z), -kWideSlack, z);
   w.hx = __builtin_fmaf(__builtin_fabsf(x), kWideSlack, x);
   w.hy = __builtin_fmaf(__builtin_fabsf(y), kWideSlack, y);
   w.hz = __builtin_fmaf(__builtin_fabsf(z), kWideSlack, z);
   return w;
}

// The planes a ray enters and leaves through, one word per axis, child k in
// byte k.
struct WidePlanes {
   uint32_t nx, fx, ny, fy, nz, fz;
};
PTX_HD float wide_byte(uint32_t w, int k) { return (float)((w >> (8 * k)) & 255u); }

// The same planes as pairs of halves: a byte with a zero byte above it is the
// half of 2^-24 times its value, which the mixed fma (half * float + float, one
// rounding) takes as it is.  Twelve instructions make the 24 operands of a node
// that took a conversion each: a node's test has 91 VALU instructions instead
// of 105 (with the exponents kept in these units) and the path kernel spills 3
// registers instead of 9.  A 4K frame's primary rays 1,106 -> 1,087 us, 2^21
// incoherent rays 561 -> 549, 16 jobs of 2.7 M faces 47.8 -> 46.3 ms.
struct WideSteps {
   uint32_t even, odd;        // children 0 and 2, children 1 and 3
};
struct WideStepPlanes {
   WideSteps nx, fx, ny, fy, nz, fz;
};
PTX_HD WideSteps wide_steps(uint32_t w) {
   WideSteps t = {w & 0x00FF00FFu, (w >> 8) & 0x00FF00FFu};
#ifdef __HIP_DEVICE_COMPILE__
   t.odd = __builtin_amdgcn_perm(0u, w, 0x0C030C01u);
   asm("" : "+v"(t.even), "+v"(t.odd));      // or the pairs are taken apart again, an extraction a child
#endif
   return t;
}
PTX_HD WideStepPlanes wide_steps(const WidePlanes &p) {
   return WideStepPlanes{wide_steps(p.nx), wide_steps(p.fx), wide_steps(p.ny),
                         wide_steps(p.fy), wide_steps(p.nz), wide_steps(p.fz)};
}
PTX_HD float wide_step(const WideSteps &t, int k) {
   const uint32_t w = k & 1 ? t.odd : t.even;
#ifdef __HIP_DEVICE_COMPILE__
   typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
   return (float)__builtin_bit_cast(f16x2, w)[k >> 1];
#else
   return (float)(k & 2 ? w >> 16 : w & 0xFFFFu) * 0x1p-24f;
#endif
}

// Whether child k may hold a leaf that the reference visits; near is a lower
// bound (up to wide_bound) of the entry distance of everything below it.
PTX_HD float wide_bound(float t) { return __builtin_fmaf(t, kWideFar, kWideTiny); }
PTX_HD bool wide_child(const WideStepPlanes &p, int k, const WideFrame &w, float min_t, float &near) {
   const float tx = __builtin_fmaf(wide_step(p.nx, k), w.sx, w.lx), ty = __builtin_fmaf(wide_step(p.ny, k), w.sy, w.ly),
               tz = __builtin_fmaf(wide_step(p.nz, k), w.sz, w.lz);
   const float ux = __builtin_fmaf(wide_step(p.fx, k), w.sx, w.hx), uy = __builtin_fmaf(wide_step(p.fy, k), w.sy, w.hy),
               uz = __builtin_fmaf(wide_step(p.fz, k), w.sz, w.hz);
   near = fmaxf(fmaxf(fmaxf(tx, ty), tz), 0.f);
   return near <= wide_bound(fminf(fminf(fminf(ux, uy), uz), min_t));
}
PTX_HD bool wide_child(const WidePlanes &p, int k, const WideFrame &w, float min_t, float &near) {
   return wide_child(wide_steps(p), k, w, min_t, near);
}

// The same for kRaySlow rays: the reference's slab values on planes moved
// outwards by more than their rounding, in the order the signs give.  Where
// 1 / d is infinite this accepts the closed interval, which holds every box
// the reference's selections accept.
PTX_HD void wide_slow_axis(uint32_t n, uint32_t f, int k, float g, int e, float o, float i, float &near, float &far) {
   const float step = __builtin_ldexpf(1.f, e - kWideStep);
   const float a = __builtin_fmaf(wide_byte(n, k), step, g), b = __builtin_fmaf(wide_byte(f, k), step, g);
   const float ga = 4 * kWideSlack * fmaxf(__builtin_fabsf(a), __builtin_fabsf(g)),
               gb = 4 * kWideSlack * fmaxf(__builtin_fabsf(b), __builtin_fabsf(g));
   near = fmaxf(near, (i < 0 ? a + ga - o : a - ga - o) * i);
   far = fminf(far, (i < 0 ? b - gb - o : b + gb - o) * i);
}
PTX_HD bool wide_child_slow(const WidePlanes &p, int k, const Ray &r, float gx, float gy, float gz, int ex, int ey,
                            int ez, float min_t, float &near) {
   float far = kInf;
   near = 0.f;
   wide_slow_axis(p.nx, p.fx, k, gx, ex, r.ox, r.ix, near, far);
   wide_slow_axis(p.ny, p.fy, k, gy, ey, r.oy, r.iy, near, far);
   wide_slow_axis(p.nz, p.fz, k, gz, ez, r.oz, r.iz, near, far);
   return near <= wide_bound(far * kSlabScale) && near <= wide_bound(min_t);     // never past a NaN min_t
}

// The axes of direction -0 in which a leaf box that passed is flat at the
// origin's coordinate: the one test that its ancestors need not pass.
PTX_HD uint32_t wide_flat(float b0, float b1, float b2, float b3, float b4, float b5, const Ray &r) {
   return (r.ix == -kInf && b0 == r.ox && b3 == r.ox ? 1u : 0u) | (r.iy == -kInf && b1 == r.oy && b4 == r.oy ? 2u : 0u) |
          (r.iz == -kInf && b2 == r.oz && b5 == r.oz ? 4u : 0u);
}

// ---------------------------------------------------------------- traversal

// Deferred children of one lane, (reference, entry distance) each: the first
// kLds in LDS, deeper ones in the launch's spill area.  exact_trace keeps its
// one-word entries in the same memory.
template <int kLds>
struct WideStack {
   uint32_t *lds;             // __shared__ [2 * kLds * 256]: references, then distances
   u32x2 *spill;              // [max_stack - kLds][stride]
   uint32_t tid, gtid, stride, max_stack;
   __device__ __forceinline__ void put_lds(uint32_t k, uint32_t ref, float near) const {
      lds[k * 256 + tid] = ref;
      lds[(kLds + k) * 256 + tid] = __float_as_uint(near);
   }
   __device__ __forceinline__ void put(uint32_t k, uint32_t ref, float near) const {
      if (k < (uint32_t)kLds) {
         put_lds(k, ref, near);
      } else if (k < max_stack) {
         const u32x2 e = {ref, __float_as_uint(near)};
         spill[(size_t)(k - kLds) * stride + gtid] = e;
      }
   }
   __device__ __forceinline__ void get_lds(uint32_t k, uint32_t &ref, float &near) const {
      ref = lds[k * 256 + tid];
      near = __uint_as_float(lds[(kLds + k) * 256 + tid]);
   }
   __device__ __forceinline__ void sentinel() const { put_lds(0, 0xFFFFFFFFu, -kInf); }
   __device__ __forceinline__ void get(uint32_t k, uint32_t &ref, float &near) const {
      if (k < (uint32_t)kLds) {
         get_lds(k, ref, near);
      } else if (k < max_stack) {
         const u32x2 e = spill[(size_t)(k - kLds) * stride + gtid];
         ref = e.x; near = __uint_as_float(e.y);
      } else {                     // unreachable: the builder bounds the stack
         ref = 0xFFFFFFFFu; near = -kInf;
      }
   }
   __device__ __forceinline__ void put_word(uint32_t k, uint32_t v) const {
      if (k < 2u * kLds) lds[k * 256 + tid] = v;
      else if (k < 2u * max_stack)
         reinterpret_cast<uint32_t *>(spill + (size_t)(k / 2 - kLds) * stride + gtid)[k & 1u] = v;
   }
   __device__ __forceinline__ uint32_t get_word(uint32_t k) const {
      if (k < 2u * kLds) return lds[k * 256 + tid];
      return reinterpret_cast<const uint32_t *>(spill + (size_t)(k / 2 - kLds) * stride + gtid)[k & 1u];
   }
};

// Pops deferred children until one's distance is within MinT.  The lane's
// entry 0 is a sentinel (no reference, distance -inf: always within), written
// once and never overwritten, so a traversal starts at sp = 1 and ends by
// popping it.  Returns false then.
template <int kLds>
__device__ __forceinline__ bool wide_pop(Trav &s, const WideStack<kLds> &st) {
   const float m = wide_bound(s.min_t);
   float near;
   if (__builtin_amdgcn_ballot_w64(s.sp > (uint32_t)kLds) == 0) {
      do {
         s.sp--;
         st.get_lds(s.sp, s.cur, near);
         // keeps the two reads one instruction: read after the loop, the
         // reference would cost a second LDS latency
         asm("" : "+v"(s.cur), "+v"(near));
      } while (near > m);
   } else {
      do {
         s.sp--;
         st.get(s.sp, s.cur, near);
      } while (near > m);
   }
   return s.cur != 0xFFFFFFFFu;
}

// The binary records a ray falls back to.
struct BinaryScene {
   const Node64 *nodes;
   const float *tris;
   const float *root_box;
   uint32_t root_ref, root_count;
};

// The whole traversal of s.r over the binary records, in the reference's own
// steps, for the rays the wide form does not order (kWideExact).  Runs to its
// end in the calling lanes.  A deferred child is one word, its parent's index
// and side: its box is read and tested again at its pop, which gives the
// entry distance that the parent's visit gave.
template <int kLds>
__device__ __forceinline__ void exact_trace(Trav &s, const BinaryScene &b, const WideStack<kLds> &st,
                                            bool debug_pixel, bool any) {
   begin(s, b.root_box, b.root_ref, b.root_count, s.hit == 0xFFFFFFFFu ? s.min_t : kInf);
   uint32_t cur = s.cur, cnt = s.cnt, sp = 0;
   while (cur != 0xFFFFFFFFu) {
      if (cur & kLeafBit) {
         const uint32_t first = cur & ~kLeafBit;
         for (uint32_t k = 0; k < cnt; k++) {
            float v[9];
            const PTX_GLOBAL float *p = as_global(b.tris + 9 * (size_t)(first + k));
#pragma unroll
            for (int j = 0; j < 9; j++) v[j] = p[j];
            if (test_triangle(v, s.r, s.min_t, s.hu, s.hv, s.hw, debug_pixel)) {
               s.hit = first + k;
               s.after = 0;
               if (any) {
                  s.cur = 0xFFFFFFFFu;
                  st.sentinel();
                  return;
               }
            }
            s.after++;
         }
      } else {
         const Node64 *n = b.nodes + cur;
         float n0, f0, n1, f1;
         slab(n->box[0], n->box[1], n->box[2], n->box[3], n->box[4], n->box[5], s.r, n0, f0);
         slab(n->box[6], n->box[7], n->box[8], n->box[9], n->box[10], n->box[11], s.r, n1, f1);
         const bool h0 = n0 <= f0 && n0 <= s.min_t, h1 = n1 <= f1 && n1 <= s.min_t;
         const uint32_t f = (s.r.nk >> n->axis) & 1u;             // the side visited first
         const bool fh = f ? h1 : h0, sh = f ? h0 : h1;
         if (fh && sh) st.put_word(sp++, cur << 1 | (f ^ 1u));
         if (fh || sh) {
            const uint32_t side = fh ? f : f ^ 1u;
            cnt = side ? n->counts >> 16 : n->counts & 0xFFFFu;
            cur = n->ref[side];
            continue;
         }
      }
      cur = 0xFFFFFFFFu;
      while (sp > 0) {
         const uint32_t e = st.get_word(--sp), side = e & 1u;
         const Node64 *n = b.nodes + (e >> 1);
         const float *x = n->box + 6 * side;
         float near, far;
         slab(x[0], x[1], x[2], x[3], x[4], x[5], s.r, near, far);
         if (near <= s.min_t) {
            cnt = side ? n->counts >> 16 : n->counts & 0xFFFFu;
            cur = n->ref[side];
            break;
         }
      }
   }
   s.cur = 0xFFFFFFFFu;
   st.sentinel();
}

// One wide node: its four children tested, those that pass pushed so that the
// octant's first comes off the stack first, and the top popped.  Each passing
// child's place is the number of passing children visited after it, so the
// four writes need no sorting.  Returns false when the traversal has ended.
template <int kLds>
__device__ __forceinline__ bool wide_node_step(Trav &s, const WideNode *nodes, const WideStack<kLds> &st) {
   const PTX_GLOBAL u32x4 *b = reinterpret_cast<const PTX_GLOBAL u32x4 *>(
         as_global(reinterpret_cast<const char *>(nodes)) + (size_t)(s.cur << 6));
   const u32x4 head = b[0], pa = b[1], pb = b[2], pc = b[3];
   const uint32_t nk = s.r.nk;
   const float gx = __uint_as_float(head.x), gy = __uint_as_float(head.y), gz = __uint_as_float(head.z);
   const int ex = (int)(head.w << 24) >> 24, ey = (int)(head.w << 16) >> 24, ez = (int)(head.w << 8) >> 24;
   const WideFrame w = wide_frame(s.r, gx, gy, gz, ex, ey, ez);
   const bool bx = s.r.ix < 0.f, by = s.r.iy < 0.f, bz = s.r.iz < 0.f;
   const WidePlanes p = {bx ? pa.y : pa.x, bx ? pa.x : pa.y, by ? pa.w : pa.z, by ? pa.z : pa.w,
                         bz ? pb.y : pb.x, bz ? pb.x : pb.y};
   const WideStepPlanes q = wide_steps(p);
   float near[4];
   uint32_t m = 0;
#pragma unroll
   for (int k = 0; k < 4; k++) m |= wide_child(q, k, w, s.min_t, near[k]) ? 1u << k : 0u;
   if (__builtin_expect((nk & kRaySlow) != 0, 0)) {
      m = 0;
#pragma unroll
      for (int k = 0; k < 4; k++)
         m |= wide_child_slow(p, k, s.r, gx, gy, gz, ex, ey, ez, s.min_t, near[k]) ? 1u << k : 0u;
   }
   m &= head.w >> 24;
   const uint64_t order = (uint64_t)pc.z | (uint64_t)pc.w << 32;
   const uint32_t flip = (uint32_t)((int)(nk << 29) >> 31) & kLaterFlip;
   const uint32_t later = (uint32_t)(order >> ((nk >> kRayLaterShift) & 63u)) ^ flip;
   const uint32_t after = later & (m * 0x1111u);
   const uint32_t refs[4] = {pb.z, pb.w, pc.x, pc.y};
   if (__builtin_amdgcn_ballot_w64(s.sp > (uint32_t)kLds - 4u) == 0) {
      // no lane's four places pass the LDS part
#pragma unroll
      for (int k = 0; k < 4; k++)
         if (m & (1u << k)) st.put_lds(s.sp + (uint32_t)__popc(after & (15u << (4 * k))), refs[k], near[k]);
   } else {
#pragma unroll
      for (int k = 0; k < 4; k++)
         if (m & (1u << k)) st.put(s.sp + (uint32_t)__popc(after & (15u << (4 * k))), refs[k], near[k]);
   }
   s.sp += (uint32_t)__popc(m);
   return wide_pop(s, st);
}

// What a leaf that passed under a direction component of -0 is: visited, not
// reached by the reference, or for the ray to be traced again.
enum : uint32_t { kFlatVisit = 0, kFlatSkip = 1, kFlatAgain = 2 };
__device__ __forceinline__ uint32_t wide_flat_leaf(uint32_t axes, const Ray &r, const WideFace *first) {
   if (axes == 0) return kFlatVisit;
   if (r.nk & kRayLoose) return kFlatAgain;
   return axes & ~as_global(first)->flat ? kFlatSkip : kFlatVisit;
}

// One leaf step: up to two faces, the first of a leaf after its box, which is
// its header's or, for a one- or two-face leaf, the corners' own (the builder
// checks that).  With a step of its own for the header, 2^21 rays on 3,000 nested
// faces in leaves of three took 712 us instead of 628, and the longer code 16
// samples at 640x480 1,220 instead of 1,150.  Returns false when the traversal
// has ended.
template <int kLds>
__device__ __forceinline__ bool wide_leaf_step(Trav &s, const WideFace *faces, const WideLeaf *leaves,
                                               const WideStack<kLds> &st, bool debug_pixel) {
   const uint32_t kind = s.cur & ~kWideIndex;
   uint32_t idx = s.cur & kWideIndex, n = kind == kWideRaw ? s.cnt : kind == kWideTwo ? 2u : 1u;
   bool done = true;                                // this leaf is: go on with the next deferred child
   bool in = true;
   if (kind == kWideHeader) {
      const PTX_GLOBAL WideLeaf *l = as_global(leaves + idx);
      const float b0 = l->box[0], b1 = l->box[1], b2 = l->box[2], b3 = l->box[3], b4 = l->box[4], b5 = l->box[5];
      idx = l->first;
      n = l->count;
      float near, far;
      slab(b0, b1, b2, b3, b4, b5, s.r, near, far);
      in = near <= far && near <= s.min_t && n != 0;
      if (in && (s.r.nk & kRayMinus)) {
         const uint32_t what = wide_flat_leaf(wide_flat(b0, b1, b2, b3, b4, b5, s.r), s.r, faces + idx);
         in = what == kFlatVisit;
         if (what == kFlatAgain) {
            s.cur = kWideExact;
            done = false;
         }
      }
   }
   if (in) {
      typedef float f32x4 __attribute__((ext_vector_type(4)));
      const PTX_GLOBAL f32x4 *p = as_global(reinterpret_cast<const f32x4 *>(faces + idx));
      const f32x4 a = p[0], b = p[1], c = p[2];
      f32x4 d = a, e = b, g = c;
      if (n > 1) {
         d = p[3];
         e = p[4];
         g = p[5];
      }
      if (kind == kWideOne || kind == kWideTwo) {
         // vertices: (a.xyz, a.w b.xy, b.zw c.x), (d.xyz, d.w e.xy, e.zw g.x)
         float x0 = fminf(fminf(a.x, a.w), b.z), x1 = fmaxf(fmaxf(a.x, a.w), b.z);
         float y0 = fminf(fminf(a.y, b.x), b.w), y1 = fmaxf(fmaxf(a.y, b.x), b.w);
         float z0 = fminf(fminf(a.z, b.y), c.x), z1 = fmaxf(fmaxf(a.z, b.y), c.x);
         x0 = fminf(fminf(fminf(x0, d.x), d.w), e.z); x1 = fmaxf(fmaxf(fmaxf(x1, d.x), d.w), e.z);
         y0 = fminf(fminf(fminf(y0, d.y), e.x), e.w); y1 = fmaxf(fmaxf(fmaxf(y1, d.y), e.x), e.w);
         z0 = fminf(fminf(fminf(z0, d.z), e.y), g.x); z1 = fmaxf(fmaxf(fmaxf(z1, d.z), e.y), g.x);
         float near, far;
         slab(x0, y0, z0, x1, y1, z1, s.r, near, far);
         in = near <= far && near <= s.min_t;
         if (in && (s.r.nk & kRayMinus)) {
            const uint32_t what = wide_flat_leaf(wide_flat(x0, y0, z0, x1, y1, z1, s.r), s.r, faces + idx);
            in = what == kFlatVisit;
            if (what == kFlatAgain) {
               s.cur = kWideExact;
               done = false;
            }
         }
      }
      if (in) {
         const float v0[9] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x};
         if (test_triangle(v0, s.r, s.min_t, s.hu, s.hv, s.hw, debug_pixel)) {
            s.hit = idx;
            s.mesh = __float_as_uint(c.y);
            s.face = __float_as_uint(c.z);
            s.after = 0;
         }
         s.after++;
         if (n > 1) {
            const float v1[9] = {d.x, d.y, d.z, d.w, e.x, e.y, e.z, e.w, g.x};
            if (test_triangle(v1, s.r, s.min_t, s.hu, s.hv, s.hw, debug_pixel)) {
               s.hit = idx + 1;
               s.mesh = __float_as_uint(g.y);
               s.face = __float_as_uint(g.z);
               s.after = 0;
            }
            s.after++;
         }
         if (n > 2) {                                  // more faces in this leaf: the next step goes on
            s.cur = kWideRaw | (idx + 2);
            s.cnt = n - 2;
            done = false;
         }
      }
   }
   // no box passes a NaN MinT: what is deferred need not be popped one by one
   if (done && (s.r.nk & kRayHard) && s.min_t != s.min_t) s.sp = 1;
   return done ? wide_pop(s, st) : true;
}

// Lanes to gather for a step that costs the whole wave: `most`, or half of the
// lanes that hold a ray when those are few, so that the last rays of a launch,
// and the few of a small one, do not wait for lanes that never come (a 4K
// frame's primary rays 1,187 -> 1,106 us, 16 plain samples at 640x480 5.20 ->
// 4.90 ms; 3 in 8 lanes the same).
__device__ __forceinline__ uint32_t wide_gather(uint32_t most, uint32_t holding) {
   return min(most, max(1u, holding / 2u));
}

// The state a traversal starts from: s.r set up and classified, min_t = tmax.
PTX_HD void wide_begin(Trav &s, const float *root_box, uint32_t root, float tmax = kInf) {
   s.min_t = tmax;
   s.hit = 0xFFFFFFFFu;
   s.mesh = s.face = 0xFFFFFFFFu;
   s.after = 0;
   s.sp = 1;
   s.cnt = 0;
   s.hu = s.hv = s.hw = 0.f;
   float near, far;
   slab(root_box[0], root_box[1], root_box[2], root_box[3], root_box[4], root_box[5], s.r, near, far);
   s.cur = near <= far && near <= s.min_t ? root : 0xFFFFFFFFu;
}

// One leaf step, or the whole traversal over the binary records for a ray that
// needs it.  Returns false when the traversal has ended.
template <int kLds>
__device__ __forceinline__ bool wide_leaf_or_exact(Trav &s, const WideFace *faces, const WideLeaf *leaves,
                                                   const BinaryScene &b, const WideStack<kLds> &st, bool debug_pixel,
                                                   bool any) {
   if (s.cur != kWideExact) return wide_leaf_step(s, faces, leaves, st, debug_pixel);
   exact_trace(s, b, st, debug_pixel, any);
   if (s.hit != 0xFFFFFFFFu) {
      const PTX_GLOBAL WideFace *f = as_global(faces + s.hit);
      s.mesh = f->mesh;
      s.face = f->face;
   }
   return false;
}

// Runs the persistent loop.  Policy supplies:
//   kWords, words                          per-ray words beside the ray itself, and their pack / unpack
//   prepare(id, s, words)                  set up ray id in s (wide_begin), wave-wide
//   nodes(words), faces(words), leaves(words), binary(words), debug_pixel(id, words)
//   finish(id, words, s)                   write the result
// A batch of rays is set up at full width (lane j prepares ray base + j) and
// handed to the lanes that need one by lane permutes.  Node steps run until
// leaf_min lanes are at leaves or refill_min rays have ended: a leaf step costs
// about two node steps and runs for the whole wave, and a ray takes one for
// every nine or so node steps.
//
// What bounds it: VALU issue while rays remain (a node's test is 91
// instructions; 166 M wave instructions for 2^21 incoherent rays on 1.3 M
// faces, the VALU busy half of the launch's cycles at 46 % of its lanes), then
// the longest rays' chains of dependent loads.  Against the binary records (64
// bytes and two boxes a step) a ray takes half the steps, and 1,048,576 /
// 2,097,152 / 8,388,608 incoherent rays 462 / 578 / 1,516 us instead of 622 /
// 833 / 2,421; primary rays of a camera 382 / 492 / 1,194 instead of 514 / 636
// / 1,617.  Float boxes (128 bytes a node, one instruction less a plane) made
// 523 instead of 596 M instructions on a 4K frame but 27 instead of 15 lane
// loads a step: 1,772 against 1,600 us on 2^23 incoherent rays.  Five waves per
// SIMD spill 24 registers: 1,881 us.
template <int kLds, class Policy>
__device__ __forceinline__ void wide_trace(const Policy &P, const Deal &deal, uint32_t *work, uint2 *spill,
                                           uint32_t refill_min, uint32_t leaf_min, uint32_t max_stack) {
   __shared__ uint32_t lds[2 * kLds * 256];
   const uint32_t lane = __lane_id();
   const WideStack<kLds> st{lds, reinterpret_cast<u32x2 *>(spill), threadIdx.x,
                            blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x, max_stack};
   RaySource src;
   src.init(deal, work, lane);
   constexpr uint32_t kNone = 0xFFFFFFFFu;
   st.sentinel();
   Trav s;
   s.cur = kNone;
   uint32_t id = kNone;                   // the lane's ray; kNone: it has none
   typename Policy::Words words{};
   refill_min = min(refill_min, 64u);     // a wave that is all idle always refills
   // the batch being handed out: this lane's prepared ray; base, left and off are wave-uniform
   Ray g{};
   uint32_t gcur = kNone;
   typename Policy::Words gw{};
   uint32_t base = 0, left = 0, off = 0;
   while (true) {
      // lanes without a ray to step: write what has ended and take new rays,
      // when enough wait or, at the end, when all have ended
      uint64_t idle = __builtin_amdgcn_ballot_w64(s.cur == kNone);
      if ((uint32_t)__popcll(idle) >= (src.done && left == 0 ? 64u : refill_min)) {
         if (id != kNone && s.cur == kNone) {
            P.finish(id, words, s);
            id = kNone;
         }
         while (idle && !(src.done && left == 0)) {
            if (left == 0) {
               src.refill(work, lane);
               if (src.done) break;
               base = src.pool_base;
               left = src.pool_left;
               off = 0;
               src.pool_left = 0;
               if (lane < left) {
                  Trav t;
                  P.prepare(base + lane, t, gw);
                  g = t.r;
                  gcur = t.cur;
               }
            }
            const uint32_t take = min((uint32_t)__popcll(idle), left);
            const uint32_t rank = __popcll(idle & ((1ull << lane) - 1ull));
            const bool mine = ((idle >> lane) & 1ull) && rank < take;
            const uint32_t from = off + min(rank, take - 1u);
            Ray r;
            r.ox = lane_read(from, g.ox); r.oy = lane_read(from, g.oy); r.oz = lane_read(from, g.oz);
            r.dx = lane_read(from, g.dx); r.dy = lane_read(from, g.dy); r.dz = lane_read(from, g.dz);
            r.ix = lane_read(from, g.ix); r.iy = lane_read(from, g.iy); r.iz = lane_read(from, g.iz);
            r.Sx = lane_read(from, g.Sx); r.Sy = lane_read(from, g.Sy); r.Sz = lane_read(from, g.Sz);
            r.nk = lane_read(from, g.nk);
            const uint32_t cur = lane_read(from, gcur);
            const typename Policy::Words wd = P.lane_words(from, gw);
            if (mine) {
               // the state wide_begin leaves, with the root test already done
               id = base + from;
               s.r = r;
               s.min_t = kInf;
               s.hit = kNone;
               s.mesh = s.face = kNone;
               s.after = 0;
               s.sp = 1;
               s.cnt = 0;
               s.hu = s.hv = s.hw = 0.f;
               s.cur = cur;
               words = wd;
            }
            idle &= ~__builtin_amdgcn_ballot_w64(mine);
            off += take;
            left -= take;
         }
         if (!__builtin_amdgcn_ballot_w64(id != kNone) && src.done && left == 0) break;
         idle = __builtin_amdgcn_ballot_w64(s.cur == kNone);
      }
      // node steps until enough lanes are at leaves or have ended
      const bool last = src.done && left == 0;
      const uint32_t leaf_now = wide_gather(leaf_min, 64u - (uint32_t)__popcll(idle));
      while (true) {
         const bool node = (int)s.cur >= 0;
         if (!__builtin_amdgcn_ballot_w64(node)) break;
         if (node) wide_node_step(s, P.nodes(words), st);
         const uint32_t ended = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(s.cur == kNone));
         const uint32_t held = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64((int)s.cur < 0)) - ended;
         if (held >= leaf_now || (!last && ended >= refill_min)) break;
      }
      const bool leaf = (int)s.cur < 0 && s.cur != kNone;
      const uint32_t held = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(leaf));
      if (held >= leaf_now || !__builtin_amdgcn_ballot_w64((int)s.cur >= 0)) {
         if (leaf) {
            wide_leaf_or_exact(s, P.faces(words), P.leaves(words), P.binary(words), st, P.debug_pixel(id, words),
                               false);
         }
      }
   }
}
// The traversals of the calling lanes, from where wide_begin left them, to
// their ends (any: to a ray's first accepted face).
template <int kLds>
__device__ __forceinline__ void wide_run(Trav &s, const WideScene &w, const BinaryScene &b, const WideStack<kLds> &st,
                                         uint32_t leaf_min, bool debug_pixel, bool any) {
   while (true) {
      const uint32_t leaf_now = wide_gather(leaf_min, (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(s.cur != 0xFFFFFFFFu)));
      while (true) {
         const bool node = (int)s.cur >= 0;
         if (!__builtin_amdgcn_ballot_w64(node)) break;
         if (node) wide_node_step(s, w.nodes, st);
         if ((uint32_t)__popcll(__builtin_amdgcn_ballot_w64((int)s.cur < 0 && s.cur != 0xFFFFFFFFu)) >= leaf_now) break;
      }
      const bool leaf = (int)s.cur < 0 && s.cur != 0xFFFFFFFFu;
      if (!__builtin_amdgcn_ballot_w64(leaf)) {
         if (!__builtin_amdgcn_ballot_w64((int)s.cur >= 0)) return;
         continue;
      }
      if (leaf) {
         wide_leaf_or_exact(s, w.faces, w.leaves, b, st, debug_pixel, any);
         if (any && s.hit != 0xFFFFFFFFu) s.cur = 0xFFFFFFFFu;
      }
   }
}

}  // namespace dev
}  // namespace ptx
