// Device BVH traversal shared by the ray-batch kernels and the path tracer.
// One ray per lane over a BVH of width 2, 4 or 8 (node layouts in isect.h).  Hit
// children are sorted near to far; the nearest is entered and the others are
// pushed with their entry distances, so that a closest-hit query skips popped
// subtrees that start beyond its current hit.  The stack keeps its top
// `nshort` entries (kMinShort..kMaxShort, chosen at launch) in dynamic LDS,
// laid out [depth][lane] so a wave's pushes hit 64 distinct banks, and spills
// deeper entries to a private array; scene creation bounds the worst-case
// depth by kStackCapacity.  Node boxes are tested with explicit
// FMAs (they are padded outward, so the test, and the culling by entry
// distance, only have to be conservative); primitives are tested with the
// reference's exact arithmetic.
#pragma once
#include "isect.h"

namespace bgpu {
namespace trav {

// Stack entries kept in LDS per lane (the range of the launch-time choice),
// and whether entries carry their entry distance (closest-hit queries then
// skip subtrees beyond the current hit).
#ifndef BGPU_TRAV_CULL
#define BGPU_TRAV_CULL 0
#endif
constexpr int kMinShort = kMinStackLds, kMaxShort = kMaxStackLds;
constexpr bool kCull = BGPU_TRAV_CULL != 0;
// private entries beyond the shallowest LDS part
constexpr int kSpill = kStackCapacity - kMinShort;
// LDS ints per lane for nshort entries: node links, then entry distances
__host__ __device__ constexpr int lds_per_lane(int nshort) { return kCull ? 2 * nshort : nshort; }
// Dynamic LDS bytes of a traversal kernel's block.
inline size_t stack_lds_bytes(int nshort, int block) {
  return (size_t)lds_per_lane(nshort) * (size_t)block * sizeof(int);
}

// Where a lane's LDS stack entries are (entry d at lds[d * stride],
// d < nshort), and the launch's walk threshold: a wave walks inner nodes
// until every lane is at a leaf or done, or (walk > 0) until fewer than
// `walk` lanes still walk while another waits at a leaf.
struct LdsSlot {
  int* lds;
  int stride;
  int nshort;
  int walk;
};
// This lane's slot in the block's dynamic LDS (stack_lds_bytes(nshort, BLOCK)
// bytes, given at launch).
template <int BLOCK>
__device__ __forceinline__ LdsSlot lane_slot(int nshort, int walk) {
  extern __shared__ int bgpu_stack_lds[];
  return LdsSlot{bgpu_stack_lds + threadIdx.x, BLOCK, nshort, walk};
}

// The counters live in registers; only the spill arrays, which are indexed
// by the stack depth, are private memory (they belong to the caller, so that
// the compiler keeps sp and stride out of scratch).
struct Stack {
  int* lds;    // lds_per_lane(nshort) entries per lane, `stride` apart
  int stride;
  int nshort;  // entries in LDS (uniform over the launch)
  int walk;    // walk threshold of the launch (LdsSlot)
  int sp;
  int* spill_n;    // kSpill entries
  float* spill_t;  // kSpill entries when kCull
  __device__ __forceinline__ void init(const LdsSlot& s, int* sn, float* stt) {
    lds = s.lds;
    stride = s.stride;
    nshort = s.nshort;
    walk = s.walk;
    sp = 0;
    spill_n = sn;
    spill_t = stt;
  }
  __device__ __forceinline__ void push(int v, float t) {
    if (sp < nshort) {
      lds[sp * stride] = v;
      if (kCull) lds[(nshort + sp) * stride] = __float_as_int(t);
    } else {
      spill_n[sp - nshort] = v;
      if (kCull) spill_t[sp - nshort] = t;
    }
    ++sp;
  }
  __device__ __forceinline__ void pop(int* v, float* t) {
    --sp;
    // the LDS entry is read in every case (the top one when the stack is
    // deeper): a choice between the two addresses would make one generic
    // load, which occupies the address unit and waits for both memories
    const int d = sp < nshort ? sp : nshort - 1;
    *v = lds[d * stride];
    *t = kCull ? __int_as_float(lds[(nshort + d) * stride]) : 0.0f;
    if (sp >= nshort) {
      *v = spill_n[sp - nshort];
      if (kCull) *t = spill_t[sp - nshort];
    }
  }
};

// Reciprocal direction for the (padded, conservative) node boxes.  Components
// below 1e-20 in magnitude are replaced by +-1e-20 so that lo*inv - o*inv
// never forms inf - inf: the box test then sees a ray that moves 1e-20 per
// unit t along that axis, far below the box padding.
__device__ __forceinline__ float safe_rcp(float d) {
  return 1.0f / (fabsf(d) < 1e-20f ? copysignf(1e-20f, d) : d);
}

// What the node tests of one ray share: a plane x is met at x * inv - oi.
struct RayPre {
  f3 inv, oi;  // 1 / d and o / d
};
__device__ __forceinline__ RayPre ray_pre(const DRay& r) {
  const f3 inv = mk3(safe_rcp(r.d.x), safe_rcp(r.d.y), safe_rcp(r.d.z));
  return RayPre{inv, mul3(r.o, inv)};
}

__device__ __forceinline__ DRay load_ray(const DevRays& r, int i) {
  DRay ray;
  ray.o = mk3(r.ox[i], r.oy[i], r.oz[i]);
  ray.d = mk3(r.dx[i], r.dy[i], r.dz[i]);
  ray.tmin = r.tmin[i];
  ray.tmax = r.tmax[i];
  return ray;
}

// The shape tree's terms of a ray.  A plane at org + off / scale (isect.h) is
// met at t = off * a + (org * inv - o * inv); o * inv is taken 2^-22 of its size
// up for the near planes and down for the far ones, so that its own rounding
// only grows the box.  The margin covers the other roundings, and much more.
struct ShapePre {
  f3 o;
  f3 a;       // inv times the scene's 1 / scale
  f3 on, of;  // o * inv, for near and far planes
  float k;    // kSphereK0 * max sigma(o2w) sigma(w2o) (see the false-hit bound in isect.h)
  float fl;   // rounding floor: floor_k * (|o|_1 + the L1 reach of the shape boxes)
};
__device__ __forceinline__ ShapePre shape_pre(f3 o, const RayPre& rp, float inv_scale, float k, float floor_k,
                                              float reach) {
  const f3 e = mk3(fabsf(rp.oi.x) * 0x1p-22f, fabsf(rp.oi.y) * 0x1p-22f, fabsf(rp.oi.z) * 0x1p-22f);
  return ShapePre{o, scl3(rp.inv, inv_scale), add3(rp.oi, e), sub3(rp.oi, e), k,
                  floor_k * (fabsf(o.x) + fabsf(o.y) + fabsf(o.z) + reach)};
}

// The margin of a shape-tree node's children: with D = |o - org| + R an upper
// bound of |o - c| for the centre c of every shape below the node (R is the
// node's half diagonal) and h the largest of the shapes' factors,
//   max(min(k * D, kSphereK0^2 * D^2 * h), fl).
// R and h share the node's fourth word as two bfloat16, rounded up.
__device__ __forceinline__ float node_margin(f3 org, uint32_t rh, const ShapePre& sp) {
  const f3 v = sub3(sp.o, org);
  const float d2 = __builtin_fmaf(v.x, v.x, __builtin_fmaf(v.y, v.y, v.z * v.z));
  const float D = __builtin_fmaf(__builtin_amdgcn_sqrtf(d2), 1.0001f, __uint_as_float(rh & 0xffff0000u));
  const float q = kSphereK0 * kSphereK0 * 1.0001f * D * D;
  return fmaxf(fminf(sp.k * 1.0001f * D, q * __uint_as_float(rh << 16)), sp.fl);
}

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float half_of(uint32_t w, int c) {
  const half2v h = __builtin_bit_cast(half2v, w);
  return (float)(c & 1 ? h.y : h.x);
}

__device__ __forceinline__ void slab(float lx, float hx, float ly, float hy, float lz, float hz,
                                     f3 inv, f3 oi, float tmin, float tmax, bool* h, float* tn) {
  float x0 = __builtin_fmaf(lx, inv.x, -oi.x), x1 = __builtin_fmaf(hx, inv.x, -oi.x);
  float y0 = __builtin_fmaf(ly, inv.y, -oi.y), y1 = __builtin_fmaf(hy, inv.y, -oi.y);
  float z0 = __builtin_fmaf(lz, inv.z, -oi.z), z1 = __builtin_fmaf(hz, inv.z, -oi.z);
  float n = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), tmin));
  float f = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), tmax));
  *h = n <= f;
  *tn = n;
}

// Tests the W children of node `node` of the triangle tree against the ray's
// interval: lk[] the links, key[] the entry distance (finite) of the children
// that are hit and +inf for the others.
template <int W>
__device__ __forceinline__ void test_children(const float4* nodes, int node, const RayPre& rp, float tmin,
                                              float tmax, float (&key)[W], int (&lk)[W]) {
  const float4* nd = nodes + (size_t)node * (2 * W);
  float v[8 * W];
#pragma unroll
  for (int q = 0; q < (7 * W + 3) / 4; ++q) {
    const float4 x = nd[q];
    v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
  }
#pragma unroll
  for (int c = 0; c < W; ++c) {
    lk[c] = __float_as_int(v[6 * W + c]);
    bool h;
    float n;
    slab(v[c], v[W + c], v[2 * W + c], v[3 * W + c], v[4 * W + c], v[5 * W + c], rp.inv, rp.oi, tmin, tmax, &h, &n);
    key[c] = h && lk[c] != kNoChild ? fminf(n, 3.0e38f) : INFINITY;  // misses sort last
  }
}

// The same for a node of the shape tree (packed, isect.h), whose children are
// grown by the node's margin.  Near and far planes are picked by the
// direction's sign, two children at a time, so that no minimum or maximum per
// plane pair is needed, and each plane is one mixed half/float multiply-add.
template <int W>
__device__ __forceinline__ void test_shape_children(const float4* nodes, int node, const RayPre& rp, const ShapePre& sp,
                                                    float tmin, float tmax, float (&key)[W], int (&lk)[W]) {
  constexpr int Q = node_quads(W);
  // fewer than 2^27 nodes: the index fits 32 bits, the byte offset may not
  const float4* nd = nodes + (size_t)((uint32_t)node * (uint32_t)Q);
  uint32_t v[4 * Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const float4 x = nd[q];
    v[4 * q] = __float_as_uint(x.x);
    v[4 * q + 1] = __float_as_uint(x.y);
    v[4 * q + 2] = __float_as_uint(x.z);
    v[4 * q + 3] = __float_as_uint(x.w);
  }
  const f3 org = mk3(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]));
  const float pad = node_margin(org, v[3], sp);
  f3 bn = mk3(__builtin_fmaf(org.x, rp.inv.x, -sp.on.x), __builtin_fmaf(org.y, rp.inv.y, -sp.on.y),
              __builtin_fmaf(org.z, rp.inv.z, -sp.on.z));
  f3 bf = mk3(__builtin_fmaf(org.x, rp.inv.x, -sp.of.x), __builtin_fmaf(org.y, rp.inv.y, -sp.of.y),
              __builtin_fmaf(org.z, rp.inv.z, -sp.of.z));
  bn = mk3(__builtin_fmaf(-pad, fabsf(rp.inv.x), bn.x), __builtin_fmaf(-pad, fabsf(rp.inv.y), bn.y),
           __builtin_fmaf(-pad, fabsf(rp.inv.z), bn.z));
  bf = mk3(__builtin_fmaf(pad, fabsf(rp.inv.x), bf.x), __builtin_fmaf(pad, fabsf(rp.inv.y), bf.y),
           __builtin_fmaf(pad, fabsf(rp.inv.z), bf.z));
  const bool sx = rp.inv.x < 0.0f, sy = rp.inv.y < 0.0f, sz = rp.inv.z < 0.0f;
#pragma unroll
  for (int c = 0; c < W; ++c) {
    constexpr int H = W / 2;  // words of one plane set
    const uint32_t* xw = v + 4 + c / 2;
    const uint32_t* yw = xw + 2 * H;
    const uint32_t* zw = yw + 2 * H;
    const float nx = __builtin_fmaf(half_of(sx ? xw[H] : xw[0], c), sp.a.x, bn.x);
    const float fx = __builtin_fmaf(half_of(sx ? xw[0] : xw[H], c), sp.a.x, bf.x);
    const float ny = __builtin_fmaf(half_of(sy ? yw[H] : yw[0], c), sp.a.y, bn.y);
    const float fy = __builtin_fmaf(half_of(sy ? yw[0] : yw[H], c), sp.a.y, bf.y);
    const float nz = __builtin_fmaf(half_of(sz ? zw[H] : zw[0], c), sp.a.z, bn.z);
    const float fz = __builtin_fmaf(half_of(sz ? zw[0] : zw[H], c), sp.a.z, bf.z);
    const float n = fmaxf(fmaxf(fmaxf(nx, ny), nz), tmin);
    const float f = fminf(fminf(fminf(fx, fy), fz), tmax);
    lk[c] = (int)v[4 + 3 * W + c];
    const bool h = n <= f && lk[c] != kNoChild;
    key[c] = h ? __builtin_amdgcn_fmed3f(n, -3.0e38f, 3.0e38f) : INFINITY;  // misses sort last
  }
}

struct Best {
  float t, b1, b2;
  int prim;
};

// Work counts of a STATS traversal: node fetches and primitive tests, per
// tree (index 0: triangles, 1: shapes).
struct Counts {
  unsigned long long nodes[2] = {0, 0}, tests[2] = {0, 0};
};

// Compare-exchange on (key, link) pairs, ascending by key.
__device__ __forceinline__ void cex(float& ka, int& la, float& kb, int& lb) {
  const bool s = kb < ka;
  const float k0 = s ? kb : ka, k1 = s ? ka : kb;
  const int l0 = s ? lb : la, l1 = s ? la : lb;
  ka = k0; kb = k1; la = l0; lb = l1;
}
template <int W>
__device__ __forceinline__ void sort_children(float (&k)[W], int (&l)[W]) {
  if constexpr (W == 2) {
    cex(k[0], l[0], k[1], l[1]);
  } else if constexpr (W == 4) {
    cex(k[0], l[0], k[1], l[1]); cex(k[2], l[2], k[3], l[3]);
    cex(k[0], l[0], k[2], l[2]); cex(k[1], l[1], k[3], l[3]);
    cex(k[1], l[1], k[2], l[2]);
  } else {  // Batcher's odd-even merge sort of 8
    cex(k[0], l[0], k[1], l[1]); cex(k[2], l[2], k[3], l[3]);
    cex(k[4], l[4], k[5], l[5]); cex(k[6], l[6], k[7], l[7]);
    cex(k[0], l[0], k[2], l[2]); cex(k[1], l[1], k[3], l[3]);
    cex(k[4], l[4], k[6], l[6]); cex(k[5], l[5], k[7], l[7]);
    cex(k[1], l[1], k[2], l[2]); cex(k[5], l[5], k[6], l[6]);
    cex(k[0], l[0], k[4], l[4]); cex(k[1], l[1], k[5], l[5]);
    cex(k[2], l[2], k[6], l[6]); cex(k[3], l[3], k[7], l[7]);
    cex(k[2], l[2], k[4], l[4]); cex(k[3], l[3], k[5], l[5]);
    cex(k[1], l[1], k[2], l[2]); cex(k[3], l[3], k[4], l[4]);
    cex(k[5], l[5], k[6], l[6]);
  }
}

// The child to walk next (kNoChild when none is hit) after pushing the other
// hit children, the farthest first; an any-hit walk takes them as they are
// stored, since it may stop at any hit.
template <int W, bool ANY>
__device__ __forceinline__ int push_children(Stack& st, float (&key)[W], int (&lk)[W]) {
  if constexpr (ANY) {
    int next = kNoChild;
#pragma unroll
    for (int c = 0; c < W; ++c)
      if (key[c] < INFINITY) {
        if (next != kNoChild) st.push(next, 0.0f);
        next = lk[c];
      }
    return next;
  }
  sort_children<W>(key, lk);
#pragma unroll
  for (int c = W - 1; c >= 1; --c)
    if (key[c] < INFINITY) st.push(lk[c], key[c]);
  return key[0] < INFINITY ? lk[0] : kNoChild;
}

// Traverses one tree.  CLOSEST: shrinks best.t; ANY: returns at the first hit.
// EXACT (with ANY): shapes are tested with `intersect` rather than
// `intersects`, so that "any hit" is exactly "a closest hit exists".  Each
// lane visits the same nodes in the same order whatever the other lanes do;
// the wave walks inner nodes together, then tests the leaves it reached
// together (st.walk sets when the walk stops early, see LdsSlot).
template <int W, bool ANY, bool FAT, bool STATS, bool EXACT = false>
__device__ __forceinline__ bool traverse(const DevScene& sc, int root, const DRay& r, const RayPre& rp, Stack& st,
                                         Best& best, Counts& cn) {
  const ShapePre sp =
      FAT ? shape_pre(r.o, rp, sc.inv_scale, sc.shape_pad_k, sc.shape_floor_k, sc.shape_reach) : ShapePre{};
  int cur = root;  // inner node (>= 0, not kNoChild), leaf (< 0) or kNoChild (done)
  st.sp = 0;
  // the next stack entry whose subtree may still hold a hit at or before
  // best.t (an equal t can still win the tie on the primitive id), or kNoChild
  auto next = [&]() -> int {
    while (st.sp > 0) {
      int n;
      float t;
      st.pop(&n, &t);
      if (ANY || !kCull || t <= best.t) return n;
    }
    return kNoChild;
  };
  for (;;) {
    const int n_live = st.walk > 0 ? __popcll(__ballot(true)) : 0;
    while (cur >= 0 && cur != kNoChild) {
      if (st.walk > 0) {
        const int n_walk = __popcll(__ballot(true));
        if (n_walk < st.walk && n_walk < n_live) break;
      }
      if (STATS) ++cn.nodes[FAT ? 1 : 0];
      float key[W];
      int lk[W];
      const float tlim = ANY ? r.tmax : best.t;
      if (FAT) test_shape_children<W>(sc.shape_nodes, cur, rp, sp, r.tmin, tlim, key, lk);
      else test_children<W>(sc.nodes, cur, rp, r.tmin, tlim, key, lk);
      cur = push_children<W, ANY>(st, key, lk);
      if (cur == kNoChild) cur = next();
    }
    if (cur == kNoChild) break;
    if (cur < 0) {  // a leaf
      int enc = ~cur;
      int first = enc >> 4, cnt = enc & 15;
      for (int k = first; k < first + cnt; ++k) {
        const float4* pr = sc.leaf + 3 * k;
        if (STATS) ++cn.tests[FAT ? 1 : 0];
        float4 r0 = pr[0], r1 = pr[1];
        int id = __float_as_int(r0.w);
        float t, b1 = 0.0f, b2 = 0.0f;
        bool hit;
        if (!FAT) {
          float4 r2 = pr[2];
          hit = tri_test(mk3(r0.x, r0.y, r0.z), mk3(r1.x, r1.y, r1.z), mk3(r2.x, r2.y, r2.z), r.o,
                         r.d, r.tmin, ANY ? r.tmax : best.t, &t, &b1, &b2);
        } else {
          const DShape& s = sc.shapes[~__float_as_int(r1.w)];
          DRay ro;
          ro.o = xform_point(s.w2o, r.o);
          ro.d = xform_vector(s.w2o, r.d);
          ro.tmin = r.tmin;
          ro.tmax = ANY ? r.tmax : best.t;
          if (ANY && !EXACT) {
            hit = shape_intersects(s, ro);
          } else {
            int ax;
            hit = shape_intersect(s, ro, &t, &ax);
          }
        }
        if (ANY) {
          if (hit) return true;
        } else if (hit && (best.prim < 0 || t < best.t || (t == best.t && id < best.prim))) {
          best.t = t;
          best.prim = id;
          best.b1 = b1;
          best.b2 = b2;
        }
      }
      cur = next();
      if (cur == kNoChild) break;
    }
  }
  return false;
}

// The shapes of a scene without a shape tree (kFewShapes), tested with the
// walk's own arithmetic: the closest hit so far, or (EXACT as in traverse)
// whether any is hit.
template <bool STATS>
__device__ __forceinline__ void few_closest(const DevScene& sc, const DRay& r, Best& best, Counts& cn) {
  for (int s = 0; s < sc.few; ++s) {
    const DShape& sh = sc.shapes[s];
    if (STATS) ++cn.tests[1];
    DRay ro;
    ro.o = xform_point(sh.w2o, r.o);
    ro.d = xform_vector(sh.w2o, r.d);
    ro.tmin = r.tmin;
    ro.tmax = best.t;
    const int id = sc.first_shape + s;
    float t;
    int ax;
    if (shape_intersect(sh, ro, &t, &ax) && (best.prim < 0 || t < best.t || (t == best.t && id < best.prim)))
      best = Best{t, 0.0f, 0.0f, id};
  }
}
// The same before a ray's triangles are known, for walks that take rays in
// groups and finish them one by one: the shapes' closest hit up to tmax, which
// then takes the place of a triangle hit beyond it (equal distances go to the
// lower id, the triangle).  It bounds no box test: a shape in the plane of
// triangles would cull their boxes by its own rounding.
struct FewHit {
  float t;
  int prim;  // -1: none
};
template <bool STATS>
__device__ __forceinline__ FewHit few_hit(const DevScene& sc, const DRay& r, Counts& cn) {
  Best b{r.tmax, 0.0f, 0.0f, -1};
  few_closest<STATS>(sc, r, b, cn);
  return FewHit{b.t, b.prim};
}
__device__ __forceinline__ void merge(Best& best, const FewHit& s) {
  if (s.prim >= 0 && (best.prim < 0 || s.t < best.t)) best = Best{s.t, 0.0f, 0.0f, s.prim};
}
template <bool STATS, bool EXACT = false>
__device__ __forceinline__ bool few_any(const DevScene& sc, const DRay& r, Counts& cn) {
  bool found = false;
  for (int s = 0; s < sc.few; ++s) {
    const DShape& sh = sc.shapes[s];
    if (STATS && !found) ++cn.tests[1];
    DRay ro;
    ro.o = xform_point(sh.w2o, r.o);
    ro.d = xform_vector(sh.w2o, r.d);
    ro.tmin = r.tmin;
    ro.tmax = r.tmax;
    float t;
    int ax;
    found = found || (EXACT ? shape_intersect(sh, ro, &t, &ax) : shape_intersects(sh, ro));
  }
  return found;
}

template <int W, bool STATS>
__device__ __forceinline__ void closest_w(const DevScene& sc, const DRay& r, const RayPre& rp, Stack& st,
                                          Best& best, Counts& cn) {
  if (sc.tri_root >= 0) traverse<W, false, false, STATS>(sc, sc.tri_root, r, rp, st, best, cn);
  few_closest<STATS>(sc, r, best, cn);
  if (sc.shape_root >= 0) traverse<W, false, true, STATS>(sc, sc.shape_root, r, rp, st, best, cn);
}
template <int W, bool STATS, bool EXACT = false>
__device__ __forceinline__ bool any_w(const DevScene& sc, const DRay& r, const RayPre& rp, Stack& st,
                                      Counts& cn) {
  Best best{r.tmax, 0.0f, 0.0f, -1};
  if (few_any<STATS, EXACT>(sc, r, cn)) return true;
  if (sc.tri_root >= 0 && traverse<W, true, false, STATS, EXACT>(sc, sc.tri_root, r, rp, st, best, cn))
    return true;
  if (sc.shape_root >= 0 && traverse<W, true, true, STATS, EXACT>(sc, sc.shape_root, r, rp, st, best, cn))
    return true;
  return false;
}

// Closest hit over both trees (triangles, then shapes), after the root-box
// test of the accelerator primitive (Primitive/KdTree.hs:240), for a scene of
// width W.
template <int W, bool STATS, bool ROOT_INF = false>
__device__ __forceinline__ void closest_hit_w(const DevScene& sc, const DRay& r, const LdsSlot& slot,
                                              Best& best, Counts& cn) {
  best.t = r.tmax;
  best.b1 = 0.0f;
  best.b2 = 0.0f;
  best.prim = -1;
  if (ROOT_INF) {  // the root box test of the unbounded ray; r.tmax only bounds the traversal
    DRay ru = r;
    ru.tmax = INFINITY;
    if (!slab_haskell(sc.root_lo, sc.root_hi, ru)) return;
  } else if (!slab_haskell(sc.root_lo, sc.root_hi, r)) {
    return;
  }
  const RayPre rp = ray_pre(r);
  int spill_n[kSpill];
  float spill_t[kCull ? kSpill : 1];
  Stack st;
  st.init(slot, spill_n, spill_t);
  closest_w<W, STATS>(sc, r, rp, st, best, cn);
}

// Any hit (Primitive/KdTree.hs:244-246) for a scene of width W; EXACT:
// whether `intersect` (KdTree.hs:240-242) would find a hit.
template <int W, bool STATS, bool EXACT = false>
__device__ __forceinline__ bool any_hit_w(const DevScene& sc, const DRay& r, const LdsSlot& slot,
                                          Counts& cn) {
  if (!slab_haskell(sc.root_lo, sc.root_hi, r)) return false;
  const RayPre rp = ray_pre(r);
  int spill_n[kSpill];
  float spill_t[kCull ? kSpill : 1];
  Stack st;
  st.init(slot, spill_n, spill_t);
  return any_w<W, STATS, EXACT>(sc, r, rp, st, cn);
}

// Width-dispatching forms for kernels whose rays may come from scenes of
// different widths; the width is uniform per scene, so the branch is uniform
// per wave where the scene is.
template <bool STATS, bool ROOT_INF = false>
__device__ __forceinline__ void closest_hit(const DevScene& sc, const DRay& r, const LdsSlot& slot,
                                            Best& best, Counts& cn) {
  if (sc.width == 8) closest_hit_w<8, STATS, ROOT_INF>(sc, r, slot, best, cn);
  else if (sc.width == 4) closest_hit_w<4, STATS, ROOT_INF>(sc, r, slot, best, cn);
  else closest_hit_w<2, STATS, ROOT_INF>(sc, r, slot, best, cn);
}
template <bool STATS, bool EXACT = false>
__device__ __forceinline__ bool any_hit(const DevScene& sc, const DRay& r, const LdsSlot& slot,
                                        Counts& cn) {
  if (sc.width == 8) return any_hit_w<8, STATS, EXACT>(sc, r, slot, cn);
  if (sc.width == 4) return any_hit_w<4, STATS, EXACT>(sc, r, slot, cn);
  return any_hit_w<2, STATS, EXACT>(sc, r, slot, cn);
}

}  // namespace trav
}  // namespace bgpu
