// Device-side scene layout and the traversal kernel launchers.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "dev_geom.h"
#include "work_slices.h"

namespace bgpu {

// BVH node of width W (2, 4 or 8), 8 * W floats (W = 4: one 128-byte line):
//   lo.x[W] hi.x[W] lo.y[W] hi.y[W] lo.z[W] hi.z[W] link[W] h[W]
//   link >= 0: inner node; link < 0: leaf ~((first<<4)|count); kNoChild: unused
//   (unused slots repeat child 0's box and h); h: the shape tree's per-child
//   margin factor (below), 0 in the triangle tree
// This is the triangle tree's node, and what a shape-tree node is packed from
// (bvh_pack.h), to 4 + 4 * W words:
//   org.xyz (float)  the centre of the children's union box
//   R, h             bfloat16 in the high and low half of one word, rounded up:
//                    the union's half diagonal, the largest of the children's h
//   lo.x[W] hi.x[W] lo.y[W] hi.y[W] lo.z[W] hi.z[W]
//                    half precision: (plane - org) * scale, rounded outward
//   link[W]
// The planes are offsets from the node's own centre, so that half precision
// keeps 2^-11 of the node's size whatever its place in the scene; `scale` is a
// power of two per scene that maps its extent to the half range.  W = 4 takes
// 80 bytes in five loads where float planes and factors take 128 in eight: the
// traversal of scattered rays is bound by the address unit, which spends 16
// cycles and more on each 16-byte load of a wave.
// Only the shape tree is packed.  Its boxes are grown by margins of 1e-6 to
// 1e-3 of the ray's distance (below), so no rounding of a plane decides which
// shapes a ray is tested against and hits.  A triangle's box is padded by some
// 1e-5 of its size, and now and then the walk decides at its faces which of two
// triangles that share an edge is hit; with packed planes it decided otherwise
// for 20 of 2.5e8 camera rays over a million-triangle terrain, and everything
// that follows such a hit changed.  (Packed, scattered rays over 1.3 M triangles
// and 10,000 spheres took 1509 us instead of 1666, camera rays 962 instead of
// 1007, shadow segments 123 instead of 128.)
constexpr int node_words(int w) { return 4 + 4 * w; }
__host__ __device__ constexpr int node_quads(int w) { return node_words(w) / 4; }
// Leaf records, 48 B each, in leaf order:
//   r0 = (p1.xyz, prim id bits), r1 = (e1.xyz, kind bits), r2 = (e2.xyz, 0)
//   kind >= 0: triangle (e1 = p2-p1, e2 = p3-p1); kind < 0: shape index ~kind.
//
// Triangles and analytic shapes live in two BVHs sharing these arrays: the
// triangle tree is rooted at node tri_root, the shape tree at shape_root (-1
// when absent).
//
// The reference's binary32 sphere quadratic (Shape.hs:173-187, solveQuadric
// Math.hs:124-139) reports hits slightly outside the true surface, and a
// shape-tree box must contain every point it reports.  In object space, with
// u = 2^-24, the computed a = |d|^2, b = 2 o.d, c = |o|^2 - r^2 and
// b*b - (4a)*c carry an absolute error of at most 64 u |o|^2 |d|^2 in
// total, while the exact discriminant is 4 |d|^2 (r^2 - dist^2) (dist: the
// ray line's distance from the centre).  A reported hit therefore has
// dist^2 <= r^2 + 16 u |o|^2, and its t lies within 4 sqrt(u) |o| / |d| of
// the closest approach, so the hit point is within
// sqrt(r^2 + 32 u |o|^2) of the centre: an excess of at most
//   min(K0 |o|, K0^2 |o|^2 / (2 r)),  K0 = kSphereK0 >= sqrt(32 u).
// Mapped to world space with sigma(w2o) |o_world - c| >= |o| and a factor
// sigma(o2w) on distances, the children of a shape-tree node are tested
// grown by the margin computed in trav::node_margin: shape_pad_k
// (= K0 * max sigma(o2w) sigma(w2o)) bounds the first form for every shape
// kind, the factor h = sigma(o2w) sigma(w2o)^2 / (2 r) (the largest over the
// node's subtree) the second for spheres, and shape_floor_k covers the
// rounding of the ray's transform and of t.  Cylinders (the same quadratic
// in two dimensions, then range tests on the hit point), disks, quads and
// boxes keep the first form.
constexpr float kSphereK0 = 2e-3f;
// Traversal stack entries available per lane (LDS part plus private spill);
// scene creation checks the tree's worst case against it.
constexpr int kStackCapacity = 64;
// A scene of at most this many shapes has no shape tree: every ray tests them
// all, and a closest hit among them does not bound the walk of the triangles (a
// hit on a shape that lies in their plane would cull boxes by its rounding).
// The loop is uniform, so the shapes' records are scalar loads and a wave tests
// each once for all its rays, where the tree costs a second walk (a second pass
// of the refilled ray batches).  1 M rays, without and with a tree, in us:
//   scattered, 200 k triangles:   closest  any       coherent, shapes alone: closest
//     1 shape                     253 281  224 254     11.4 13.7
//     4 shapes                    266 281  226 246     16.2 16.0
//     6 shapes                    271 286  232 255     19.4 18.0
//     8 shapes                    281 292  243 257     23.6 19.7
// Scattered rays over shapes alone still gain at eight (51 and 74); the line
// lies at six because of coherent ones.
constexpr int kFewShapes = 6;
// link of an unused child slot in a node
constexpr int32_t kNoChild = 0x7fffffff;

struct DevScene {
  const float4* nodes;        // triangle tree, 2 * width float4 per node
  const float4* shape_nodes;  // shape tree, node_quads(width) float4 per node
  const float4* leaf;
  const DShape* shapes;
  float root_lo[3], root_hi[3];
  int32_t tri_root;    // -1 if no triangles
  int32_t shape_root;  // -1 if no shapes
  float shape_pad_k;    // K0 * max sigma(o2w) sigma(w2o) over the shapes
  int32_t num_nodes;
  int32_t width;        // 2, 4 or 8 children per node
  float shape_floor_k;  // rounding term of the shape margins
  float shape_reach;    // L1 norm of the shape tree's farthest corner from the world origin
  float inv_scale;      // 1 / scale of the packed planes
  int32_t few;          // shapes tested one by one, without a tree (kFewShapes), else 0
  int32_t first_shape;  // primitive id of shape 0
};

struct DevRays {
  const float *ox, *oy, *oz, *dx, *dy, *dz, *tmin, *tmax;
};
struct DevHits {
  float *t, *b1, *b2;
  int32_t* prim;
};

// Launch-shape knobs chosen by the autotuner.
struct TraceConfig {
  int block = 256;
  int persistent = 1;  // lanes refill with new rays (1) or one ray per thread (0)
  int stack = 12;      // traversal stack entries per lane kept in LDS
  int refill = 32;     // lane refill: idle lanes that trigger it (1..64)
  int walk = 16;       // walk inner nodes while at least this many lanes do (0: until all are at leaves)
};
// The range of TraceConfig::stack (and of the bounce loop's pt.stack); deeper
// entries spill to private memory.
constexpr int kMinStackLds = 8, kMaxStackLds = 24;

// The persistent passes take their items from kWorkCounters counters, a
// 128-byte line each; a launch has two passes.
constexpr int kCounterStride = 32;
constexpr int kWorkWords = 2 * (int)kWorkCounters * kCounterStride;
// Words of the per-GPU scratch array of the allocation-free ray batches: the
// passes' counters, then the four 64-bit work counters of BGPU_COUNT.
// scratch_address returns its device address on the current device.
constexpr int kScratchWords = kWorkWords + 64;
hipError_t scratch_address(void** ptr);
// Zeroes n 32-bit words on stream s with a kernel.
hipError_t zero_words(unsigned int* p, int n, hipStream_t s);

// `work`: kWorkWords words for the persistent kernels' counters, zeroed by the
// launch (may be null, which selects one ray per thread).
hipError_t launch_closest(const DevScene& sc, const DevRays& r, int n, const DevHits& h,
                          const TraceConfig& cfg, hipStream_t s, unsigned long long* counters,
                          unsigned int* work);
hipError_t launch_any(const DevScene& sc, const DevRays& r, int n, uint8_t* occ,
                      const TraceConfig& cfg, hipStream_t s, unsigned long long* counters,
                      unsigned int* work);

}  // namespace bgpu
