// Device-side tree traversal and triangle test shared by the visibility,
// transfer and direct-light kernels.  gfx950, wave64.
//
// Built with -ffp-contract=off: the triangle test below rounds once per
// operation in the same association as the CPU restatement, so hit index and
// hit t are bit-identical to it.  Traversal arithmetic only culls, with
// conservative bounds, so its rounding never changes a result.  The optimised
// path walks a 4-wide bounding-volume hierarchy (BvhTracer, built by bvh.hip),
// the plain path the kd-tree (KdTracer).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace vr {

struct DevScene {
  // kd-tree (plain path)
  const uint2 *nodes;     // x = children ((index << 2) | type), y = split bits
  const float4 *refs;     // 3 float4 per leaf reference (leaf order)
  const float4 *planes;   // per triangle (nx, ny, nz, d), original order
  float bmin[3], bmax[3];
  float M;                // max(1, max |scene coordinate|)
  int has_sky;
  int empty;              // no triangles
  // a second tree over the TRACE_ID_SKY triangles alone (when has_sky)
  const uint2 *sky_nodes;
  const float4 *sky_refs;
  float sky_bmin[3], sky_bmax[3];
  // 4-wide hierarchies over all triangles and over the sky triangles (null:
  // no triangle of theirs can be hit): 8 float4 per node (the children's min x,
  // max x, min y, max y, min z, max z, child words, unused) and 3 float4 per
  // triangle, each triangle once
  const float4 *bvh, *bvh_refs;
  const float4 *sky_bvh, *sky_bvh_refs;
  int has_bvh;            // 0: too large for 32-bit node offsets, walk the kd-tree
};

// Child words of the hierarchy: an inner node's index, or a leaf: kBvhLeaf, a
// triangle count and the first triangle's record (a leaf of no triangles: no
// child).
constexpr uint32_t kBvhLeaf = 0x80000000u;
constexpr int kBvhCntShift = 28;
constexpr uint32_t kBvhFirstMask = (1u << kBvhCntShift) - 1u;
// Stack entries of a walk: it leaves at most three children per level, and the
// build keeps the tree within kBvhStack / 3 levels.
constexpr int kBvhStack = 64;

constexpr float kTiny = 1e-20f;

// Workgroups are dispatched round-robin over the 8 XCDs of an MI355X, each
// with its own L2.  Remap workgroup b of nb so that XCD x takes one
// contiguous range of work chunks: neighbouring rays (same origin patch in a
// MakeTransfers batch) then share one L2.  A bijection on [0, nb).
__device__ __forceinline__ uint32_t xcd_chunk(uint32_t b, uint32_t nb) {
  const uint32_t x = b & 7u, k = b >> 3, per = nb >> 3, rem = nb & 7u;
  return x * per + min(x, rem) + k;
}
// The same with the work dealt to the XCDs in groups of g consecutive
// chunks, round-robin (group q to XCD q mod 8), so that an XCD whose
// contiguous range would hold more work than the others' does not set the
// launch's end; chunks of a group stay on one XCD.  g = 0 is xcd_chunk.  The
// blocks past the last whole round of 8 g take xcd_chunk over the rest.
// A bijection on [0, nb).  On the 8x8-room level, with the hierarchy: PVS
// MakeTransfers 217.6 ms with one range per XCD, 181.5 with groups of 256
// chunks, 179 with 16 or 64, 199 with 4096; a TestLine batch of 4 M segments
// 275, 281, 257 and 283 us; closest hits 182-185 us with any of them.
constexpr uint32_t kXcdGroup = 256;
__device__ __forceinline__ uint32_t xcd_group_chunk(uint32_t b, uint32_t nb, uint32_t g) {
  if (g == 0) return xcd_chunk(b, nb);
  const uint32_t full = nb / (8u * g) * (8u * g);
  if (b >= full) return full + xcd_chunk(b - full, nb - full);
  const uint32_t x = b & 7u, k = b >> 3;
  return ((k / g) * 8u + x) * g + k % g;
}
constexpr uint32_t kTriMask = (1u << 28) - 1u;

__device__ __forceinline__ float sel3(int c, float a, float b, float d) {
  return c == 0 ? a : (c == 1 ? b : d);
}

// Projected-barycentric hit test (frozen semantics of Trace4Rays, which is a
// stub at raytracer/environment.go:140-145): accept t in [tmin, tbest),
// equal t resolved to the lower triangle index.  SKIPSKY ignores
// TRACE_ID_SKY triangles.
template <bool SKIPSKY = false>
__device__ __forceinline__ void tri_test(const float4 *__restrict__ refs, uint32_t k, float ox,
                                         float oy, float oz, float dx, float dy, float dz,
                                         float tmin, int32_t skip, float &tbest, int32_t &best,
                                         int32_t &best_id, uint32_t &best_ref) {
  const float4 q0 = refs[3 * (size_t)k + 0];
  const float4 q1 = refs[3 * (size_t)k + 1];
  const float4 q2 = refs[3 * (size_t)k + 2];
  const int32_t id = __float_as_int(q2.z);
  if (id == skip) return;
  if (SKIPSKY && (id & 0x01000000)) return;
  const uint32_t meta = __float_as_uint(q2.w);
  const int32_t tri = (int32_t)(meta & kTriMask);
  const float den = (q0.x * dx + q0.y * dy) + q0.z * dz;
  if (!(den != 0.0f)) return;
  const float num = q0.w - ((q0.x * ox + q0.y * oy) + q0.z * oz);
  const float t = num / den;
  if (!(t >= tmin && (t < tbest || (t == tbest && tri < best)))) return;
  const int c0 = (int)((meta >> 28) & 3u), c1 = (int)(meta >> 30);
  const float h0 = sel3(c0, ox, oy, oz) + t * sel3(c0, dx, dy, dz);
  const float h1 = sel3(c1, ox, oy, oz) + t * sel3(c1, dx, dy, dz);
  const float b0 = (q1.x * h0 + q1.y * h1) + q1.z;
  const float b1 = (q1.w * h0 + q2.x * h1) + q2.y;
  if (b0 >= 0.0f && b1 >= 0.0f && (b0 + b1) <= 1.0f) {
    tbest = t;
    best = tri;
    best_id = id;
    best_ref = k;
  }
}
constexpr uint32_t kNoRef = 0xffffffffu;

// kd nodes a scene may hold (24-bit indices; the scene build checks)
constexpr uint32_t kStackNodeBits = 24;

// Traversal stack of the hierarchy's walk: the first S entries of a lane in
// LDS (entry k of lane l at [64 k + l]: conflict free), deeper ones in private
// scratch.  The deeper entries live in a separate object (BvhSpill) the stack
// points to: an array indexed at run time sits in private memory, and keeping
// it out of this struct lets the LDS pointer stay in a register.  E: 4-byte
// child words, or 8 bytes with the entry's key (BvhTracer::walk).
template <int S, class E>
struct BvhSpill {
  E v[kBvhStack - S];
};
#define VR_PRIVATE __attribute__((address_space(5)))
template <int S, class E>
struct BvhLaneStack {
  E *e;              // this lane's entry 0 in LDS
  VR_PRIVATE E *pv;  // private-memory pointer: scratch (not flat) accesses
  __device__ BvhLaneStack(E *lds, int lane, BvhSpill<S, E> &sp)
      : e(lds + lane), pv((VR_PRIVATE E *)sp.v) {}
  __device__ void push(int sp, E v) {
    if (sp < S) e[64 * sp] = v;
    else pv[sp - S] = v;
  }
  __device__ E get(int sp) const {
    if (sp < S) return e[64 * sp];
    return pv[sp - S];
  }
};

template <int D>
struct ScratchStack {
  uint32_t node[D];
  float a[D], b[D];
  __device__ void push(int sp, uint32_t n, float x, float y) {
    node[sp] = n;
    a[sp] = x;
    b[sp] = y;
  }
  __device__ void get(int sp, uint32_t &n, float &x, float &y) const {
    n = node[sp];
    x = a[sp];
    y = b[sp];
  }
};

// Interval bounds in the walk are compared as int32 bit patterns: one
// v_min_i32 / v_max_i32, with no NaN quieting of loop-carried values.  For
// two non-negative floats, or one of each sign, this is the float min / max;
// for two negatives (only when a caller's tmin < 0) "min" returns the larger
// and "max" the smaller, so an upper bound (min) only grows and a lower
// bound (max) only shrinks: intervals widen, the walk visits more, and the
// result is unchanged.
__device__ __forceinline__ float tmin_wide(float a, float b) {
  return __int_as_float(min(__float_as_int(a), __float_as_int(b)));
}
__device__ __forceinline__ float tmax_wide(float a, float b) {
  return __int_as_float(max(__float_as_int(a), __float_as_int(b)));
}

// What a walk needs of its ray besides origin and direction, the same for
// every tree of a scene (the margin dl depends on the scene's extent M):
// the reciprocal direction, and the slab terms of a split plane s on axis a,
//   t = ((s +- dl) - o_a) i_a = s i_a + (+-dl - o_a) i_a,
// the near child's exit with +dl toward the ray (copysign(dl, i_a)), the far
// child's entry with -dl; the terms after s i_a are fixed per ray, and their
// rounding (and the fma's) stays far inside the dl margin.  A segment that
// walks the sky tree and then the full tree computes this once.
struct RayPre {
  float ix, iy, iz, dl, ex, ey, ez, fx, fy, fz;
};
__device__ __forceinline__ RayPre ray_pre(float M, float ox, float oy, float oz, float dx,
                                          float dy, float dz) {
  RayPre r;
  const float om = fmaxf(fabsf(ox), fmaxf(fabsf(oy), fabsf(oz)));
  r.dl = (M + om) * 0x1p-15f;
  r.ix = 1.0f / (fabsf(dx) < kTiny ? copysignf(kTiny, dx) : dx);
  r.iy = 1.0f / (fabsf(dy) < kTiny ? copysignf(kTiny, dy) : dy);
  r.iz = 1.0f / (fabsf(dz) < kTiny ? copysignf(kTiny, dz) : dz);
  r.ex = (copysignf(r.dl, r.ix) - ox) * r.ix;
  r.fx = (-copysignf(r.dl, r.ix) - ox) * r.ix;
  r.ey = (copysignf(r.dl, r.iy) - oy) * r.iy;
  r.fy = (-copysignf(r.dl, r.iy) - oy) * r.iy;
  r.ez = (copysignf(r.dl, r.iz) - oz) * r.iz;
  r.fz = (-copysignf(r.dl, r.iz) - oz) * r.iz;
  return r;
}

// Walks one kd-tree (nodes/refs/bounds) for hits with tmin <= t < tmax that
// come before (tbest, best) in (t, triangle index) order, updating them; the
// result is the first of the hits in that order, bit for bit the brute-force
// result.  The plain path and scenes past the hierarchy's node limit take this
// walk.  ANY: return at the first accepted hit.  SKIPSKY: ignore TRACE_ID_SKY
// triangles.  POSTPONE (closest hits): lanes hold their next leaf and walk on
// until every lane of the wave holds one (below).  Returns whether a hit was
// accepted (best_ref = its leaf-reference index).  D = stack capacity; the host
// guarantees tree depth < D.
template <int D, bool ANY, bool SKIPSKY, bool POSTPONE, class Stack>
__device__ bool walk_tree(const uint2 *__restrict__ nodes, const float4 *__restrict__ refs,
                          const float *bmin, const float *bmax, const RayPre &rp, Stack &st,
                          float ox, float oy, float oz, float dx, float dy, float dz,
                          float tmin, float tmax, int32_t skip, float &tbest, int32_t &best,
                          int32_t &best_id, uint32_t &best_ref) {
  static_assert(!(ANY && POSTPONE), "any-hit walks return at their first leaf's hit");
  const int32_t best0 = best;
  const float dl = rp.dl, ix = rp.ix, iy = rp.iy, iz = rp.iz;
  float ta = tmin, tb = tmax;
  {
    float t1 = ((bmin[0] - dl) - ox) * ix, t2 = ((bmax[0] + dl) - ox) * ix;
    ta = fmaxf(ta, fminf(t1, t2));
    tb = fminf(tb, fmaxf(t1, t2));
    t1 = ((bmin[1] - dl) - oy) * iy;
    t2 = ((bmax[1] + dl) - oy) * iy;
    ta = fmaxf(ta, fminf(t1, t2));
    tb = fminf(tb, fmaxf(t1, t2));
    t1 = ((bmin[2] - dl) - oz) * iz;
    t2 = ((bmax[2] + dl) - oz) * iz;
    ta = fmaxf(ta, fminf(t1, t2));
    tb = fminf(tb, fmaxf(t1, t2));
  }
  if (!(ta <= tb)) return false;
  // An any-hit walk returns at its first accepted hit, so tbest is fixed
  // while it runs: clamping tb to it here leaves every min(tb, tbest) of
  // the walk unchanged (an integer-order min, associative), and a stacked
  // entry, pushed only when its start is at most that bound, never needs
  // the pop's prune.
  if constexpr (ANY) tb = tmin_wide(tb, tbest);
  const float ex = rp.ex, ey = rp.ey, ez = rp.ez, fx = rp.fx, fy = rp.fy, fz = rp.fz;
  int sp = 0;
  uint32_t node = 0;
  // next stacked node whose interval can still hold a hit before tbest
  auto pop = [&]() -> bool {
    while (sp > 0) {
      --sp;
      float a, b;
      uint32_t n;
      st.get(sp, n, a, b);
      if (!ANY && a > tbest) continue;
      node = n;
      ta = a;
      tb = b;
      return true;
    }
    return false;
  };
  if constexpr (POSTPONE) {
    // "while-while" with postponed leaves: a lane descends through inner
    // nodes and empty leaves to its next leaf holding triangles and keeps it;
    // until every lane of the wave holds one, a lane that already does walks
    // on to its next such leaf and stops there.  Then the wave tests the held
    // leaves together.  Visits differ from a depth-first walk only in order
    // and, for a closest hit, in leaves tested before a hit found later would
    // have pruned them; the result is the least hit in (t, triangle) order
    // either way.  A step assigns each loop value once, by selects, and the
    // push is a predicated store.  Closest hits take this walk: their long
    // walks through many leaves keep more lanes busy.  Any-hit walks, which
    // mostly end at their first leaf, do not.
    uint32_t lstart = 0, lcnt = 0;  // the held leaf's triangles (none: lcnt 0)
    bool live = true;               // node, ta, tb: the next node to visit
    for (;;) {
      uint2 nd = nodes[node];
      for (;;) {
        if ((nd.x & 3u) == 3u) {
          const uint32_t c = (uint32_t)__uint_as_float(nd.y);
          if (c != 0u) {
            if (lcnt != 0u) break;  // a second leaf: visit it after the held one
            lstart = nd.x >> 2;
            lcnt = c;
          }
          if (!pop()) {
            live = false;
            break;
          }
        } else {
          const uint32_t type = nd.x & 3u;
          const float sv = __uint_as_float(nd.y);
          const float i_a = sel3((int)type, ix, iy, iz);
          const float near_end = __builtin_fmaf(sv, i_a, sel3((int)type, ex, ey, ez));
          const float far_start = __builtin_fmaf(sv, i_a, sel3((int)type, fx, fy, fz));
          const uint32_t left = nd.x >> 2;
          const bool fwd = i_a >= 0.0f;
          const uint32_t near_n = fwd ? left : left + 1, far_n = fwd ? left + 1 : left;
          const float tbe = tmin_wide(tb, tbest);
          const bool near_ok = ta <= tmin_wide(near_end, tbe);
          const float fs = tmax_wide(far_start, ta);
          const bool far_ok = fs <= tbe;
          // the stack holds at most one entry per level of the path to the
          // current node, and the host checks tree depth < D
          if (near_ok && far_ok) {
            st.push(sp, far_n, fs, tb);
            ++sp;
          }
          node = near_ok ? near_n : far_n;
          const float tb_near = tmin_wide(tb, near_end);
          ta = near_ok ? ta : fs;
          tb = near_ok ? tb_near : tb;
          if (!near_ok && !far_ok && !pop()) {
            live = false;
            break;
          }
        }
        nd = nodes[node];
        if (__ballot(lcnt == 0u) == 0) break;  // every walking lane holds a leaf
      }
      for (uint32_t k = lstart; k < lstart + lcnt; ++k)
        tri_test<SKIPSKY>(refs, k, ox, oy, oz, dx, dy, dz, tmin, skip, tbest, best, best_id,
                          best_ref);
      lcnt = 0u;
      if (!live) break;
    }
  } else {
    // "while-while": a lane descends through inner nodes to its next leaf
    // before the wave tests leaves, so lanes test triangles together.  Each
    // lane visits the same nodes in the same order as one step per iteration.
    // A step assigns each loop value once, by selects, and the push is a
    // predicated store.  A step where neither child can hold a hit leaves the
    // descent as an empty leaf: the pop that follows every leaf continues the
    // walk, as a pop right there would.
    constexpr uint2 kEmptyLeaf = {3u, 0u};  // leaf, no triangles
    for (;;) {
      uint2 nd = nodes[node];
      while ((nd.x & 3u) != 3u) {
        const uint32_t type = nd.x & 3u;
        const float sv = __uint_as_float(nd.y);
        const float i_a = sel3((int)type, ix, iy, iz);
        const float near_end = __builtin_fmaf(sv, i_a, sel3((int)type, ex, ey, ez));
        const float far_start = __builtin_fmaf(sv, i_a, sel3((int)type, fx, fy, fz));
        const uint32_t left = nd.x >> 2;
        const bool fwd = i_a >= 0.0f;
        const uint32_t near_n = fwd ? left : left + 1, far_n = fwd ? left + 1 : left;
        const float tbe = ANY ? tb : tmin_wide(tb, tbest);
        const bool near_ok = ta <= tmin_wide(near_end, tbe);
        const float fs = tmax_wide(far_start, ta);
        const bool far_ok = fs <= tbe;
        // the stack holds at most one entry per level of the path to the
        // current node, and the host checks tree depth < D
        if (near_ok && far_ok) {
          st.push(sp, far_n, fs, tb);
          ++sp;
        }
        node = near_ok ? near_n : far_n;
        const float tb_near = tmin_wide(tb, near_end);
        ta = near_ok ? ta : fs;
        tb = near_ok ? tb_near : tb;
        if (!near_ok && !far_ok) {
          nd = kEmptyLeaf;
          break;
        }
        nd = nodes[node];
      }
      const uint32_t start = nd.x >> 2;
      const uint32_t cnt = (uint32_t)__uint_as_float(nd.y);
      for (uint32_t k = start; k < start + cnt; ++k)
        tri_test<SKIPSKY>(refs, k, ox, oy, oz, dx, dy, dz, tmin, skip, tbest, best, best_id,
                          best_ref);
      if (ANY && best != best0) return true;
      if (!pop()) break;
    }
  }
  return best != best0;
}

// ---- tracers: one ray against the scene's trees ---------------------------
// A tracer is set up for a ray (begin) and then walks the full tree or the sky
// tree for hits with tmin <= t that come before (tbest, best) in (t, triangle
// index) order, updating them; ANY: it returns at the first accepted hit.
// Returns whether a hit was accepted (ref = its record's index).

template <int D>
struct KdTracer {
  const DevScene &sc;
  ScratchStack<D> &st;  // not a member: the ray would move to private memory with it
  RayPre rp;
  float ox, oy, oz, dx, dy, dz;
  __device__ KdTracer(const DevScene &s, ScratchStack<D> &stack) : sc(s), st(stack) {}
  __device__ __forceinline__ void begin(float ox_, float oy_, float oz_, float dx_, float dy_,
                                        float dz_) {
    ox = ox_;
    oy = oy_;
    oz = oz_;
    dx = dx_;
    dy = dy_;
    dz = dz_;
    rp = ray_pre(sc.M, ox, oy, oz, dx, dy, dz);
  }
  template <bool ANY, bool SKIPSKY>
  __device__ __forceinline__ bool full(float tmin, int32_t skip, float &tbest, int32_t &best,
                                       int32_t &id, uint32_t &ref) {
    return walk_tree<D, ANY, SKIPSKY, !ANY>(sc.nodes, sc.refs, sc.bmin, sc.bmax, rp, st, ox, oy,
                                            oz, dx, dy, dz, tmin, tbest, skip, tbest, best, id,
                                            ref);
  }
  template <bool ANY>
  __device__ __forceinline__ bool sky(float tmin, int32_t skip, float &tbest, int32_t &best,
                                      int32_t &id, uint32_t &ref) {
    return walk_tree<D, ANY, false, false>(sc.sky_nodes, sc.sky_refs, sc.sky_bmin, sc.sky_bmax,
                                           rp, st, ox, oy, oz, dx, dy, dz, tmin, tbest, skip,
                                           tbest, best, id, ref);
  }
};

// The 4-wide hierarchy.  Bound by issue and by the vector cache: a node is
// 112 bytes per lane (7 loads) and some 80 vector instructions.  On the
// 8x8-room level a wave of 64 MakeTransfers segments takes 14-18 node steps
// and 1-2 triangle tests (counted on the CPU; the kd-tree took 60-140 and
// 40-110).
//
// A child's slab entry is fma(near plane, 1/d, a) with a = -o/d (and the exit
// alike), the near plane picked by the direction's sign through the load's
// offset.  The boxes hold every point an accepted hit can lie at for origins
// within the scene's extent M, with the slab arithmetic's rounding
// (k_bvh_bounds); an origin farther out widens the slabs by 96 u (|o| - M)
// here.  A direction component of 0 counts as +-1e-20.
//
// While the wave's walking lanes are at the same node (most steps near the
// root for rays that start close together), the node comes through scalar
// loads: a vector load of one address still takes the vector cache 16 cycles,
// 112 per node, which was 81 % busy on the level's TestLine batch.  Lanes of
// several octants then sort each axis's two times, 24 instructions more: with
// one octant alone (about half of MakeTransfers' waves) the level's pair trace
// took 186 ms against 166, the closest hits 205 us against 188.
//
// A wave that walks as one (a node visited when any of its rays enters it,
// nothing but scalar loads, the stack in a register) was slower: 28 steps for
// 64 pair segments and 3100 instead of 1250 vector instructions, 300 ms.
typedef uint32_t u32v4 __attribute__((ext_vector_type(4)));
typedef float f32v4 __attribute__((ext_vector_type(4)));
struct Planes {
  f32v4 ax, bx, ay, by, az, bz;  // the four children's near and far planes, by axis
  u32v4 ch;                      // their words
  template <class P>
  __device__ __forceinline__ void load(P pax, P pbx, P pay, P pby, P paz, P pbz, P pch) {
    auto f = [](P p) {
      if constexpr (std::is_same<P, const char *>::value)
        return *reinterpret_cast<const f32v4 *>(p);
      else  // constant address space: scalar loads
        return *(const __attribute__((address_space(4))) f32v4 *)p;
    };
    ax = f(pax);
    bx = f(pbx);
    ay = f(pay);
    by = f(pby);
    az = f(paz);
    bz = f(pbz);
    const f32v4 c = f(pch);
    ch = u32v4{__float_as_uint(c.x), __float_as_uint(c.y), __float_as_uint(c.z),
               __float_as_uint(c.w)};
  }
};
template <int S, class E>
struct BvhTracer {
  static constexpr bool kKeyed = sizeof(E) == 8;  // stack entries with keys: closest hits
  const DevScene &sc;
  BvhLaneStack<S, E> st;
  float ox, oy, oz, dx, dy, dz;
  float ix, iy, iz, nx, ny, nz, fx, fy, fz;
  uint32_t sx, sy, sz;  // byte offset of the near planes in a node, by axis
  bool uni;             // scalar node loads will do (all rays set up together): one
                        // octant, or no origin beyond M (nx == fx, so that either
                        // plane of an axis can be the near one)
  __device__ BvhTracer(const DevScene &s, E *lds, int lane, BvhSpill<S, E> &sp)
      : sc(s), st(lds, lane, sp) {}
  __device__ __forceinline__ void begin(float ox_, float oy_, float oz_, float dx_, float dy_,
                                        float dz_) {
    ox = ox_;
    oy = oy_;
    oz = oz_;
    dx = dx_;
    dy = dy_;
    dz = dz_;
    const float om = fmaxf(fabsf(ox), fmaxf(fabsf(oy), fabsf(oz)));
    const float e = fmaxf(om - sc.M, 0.0f) * (96.0f * 0x1p-24f);
    ix = 1.0f / (fabsf(dx) < kTiny ? copysignf(kTiny, dx) : dx);
    iy = 1.0f / (fabsf(dy) < kTiny ? copysignf(kTiny, dy) : dy);
    iz = 1.0f / (fabsf(dz) < kTiny ? copysignf(kTiny, dz) : dz);
    nx = (-copysignf(e, ix) - ox) * ix;
    ny = (-copysignf(e, iy) - oy) * iy;
    nz = (-copysignf(e, iz) - oz) * iz;
    fx = (copysignf(e, ix) - ox) * ix;
    fy = (copysignf(e, iy) - oy) * iy;
    fz = (copysignf(e, iz) - oz) * iz;
    sx = (__float_as_uint(ix) >> 31) << 4;
    sy = (__float_as_uint(iy) >> 31) << 4;
    sz = (__float_as_uint(iz) >> 31) << 4;
    const uint32_t o = sx | (sy << 1) | (sz << 2);
    uni = __ballot(o != (uint32_t)__builtin_amdgcn_readfirstlane((int)o)) == 0 ||
          __ballot(e != 0.0f) == 0;
  }
  template <bool ANY, bool SKIPSKY>
  __device__ __forceinline__ bool full(float tmin, int32_t skip, float &tbest, int32_t &best,
                                       int32_t &id, uint32_t &ref) {
    return walk<ANY, SKIPSKY>(sc.bvh, sc.bvh_refs, tmin, skip, tbest, best, id, ref);
  }
  template <bool ANY>
  __device__ __forceinline__ bool sky(float tmin, int32_t skip, float &tbest, int32_t &best,
                                      int32_t &id, uint32_t &ref) {
    return walk<ANY, false>(sc.sky_bvh, sc.sky_bvh_refs, tmin, skip, tbest, best, id, ref);
  }

  // Depth first.  Without keys (any hit; and the closest hit in the sky tree
  // of a few dozen triangles) the children are taken in node order: sorting
  // them changed an any-hit wave's steps by less than 5 % on six batches.
  // With keys (closest hits) they are sorted by entry distance, which a popped
  // entry is checked against again: 27 instead of 82 steps per wave of
  // hemisphere rays.  A key is the entry distance with the child's number in
  // its two low bits (rounded down; entries at or behind t = 0 have distance
  // bits 0 and are never skipped).
  template <bool ANY, bool SKIPSKY>
  __device__ __forceinline__ bool walk(const float4 *__restrict__ nodes,
                                       const float4 *__restrict__ refs, float tmin, int32_t skip,
                                       float &tbest, int32_t &best, int32_t &best_id,
                                       uint32_t &best_ref) {
    // no t lies in an empty interval, and no hit has a NaN in its ray: without
    // this such a ray would enter every box
    if (!nodes || (best < 0 && !(tmin < tbest)) || __builtin_isunordered(ox, oy) ||
        __builtin_isunordered(oz, dx) || __builtin_isunordered(dy, dz))
      return false;
    const int32_t best0 = best;
    const char *const base = reinterpret_cast<const char *>(nodes);
    constexpr uint32_t kDone = 0xffffffffu;  // no stacked entry is left
    uint32_t cur = 0;
    int sp = 0;
    auto pop = [&]() -> uint32_t {
      if constexpr (kKeyed) {
        while (sp > 0) {
          const uint64_t w = st.get(--sp);
          const uint32_t key = (uint32_t)(w >> 32);
          if (key < 4u || __uint_as_float(key & ~3u) <= tbest) return (uint32_t)w;
        }
        return kDone;
      } else {
        --sp;
        if (__ballot(sp >= S) == 0) return st.e[64 * sp];
        return st.get(sp);
      }
    };
    if constexpr (!kKeyed) st.push(sp++, kDone);  // the last entry popped
    // the children a ray enters: the next one to visit, the others stacked
    auto take = [&](bool h0, bool h1, bool h2, bool h3, float t0, float t1, float t2, float t3,
                    const u32v4 &ch) -> uint32_t {
      if constexpr (kKeyed) {
        constexpr uint32_t kMiss = 0xffffffffu;
        auto key = [](bool h, float t, uint32_t k) {
          return h ? (__float_as_uint(fmaxf(t, 0.0f)) & ~3u) | k : kMiss;
        };
        uint32_t k0 = key(h0, t0, 0u), k1 = key(h1, t1, 1u), k2 = key(h2, t2, 2u),
                 k3 = key(h3, t3, 3u);
        auto order = [](uint32_t &a, uint32_t &b) {
          const uint32_t lo = min(a, b), hi = max(a, b);
          a = lo;
          b = hi;
        };
        order(k0, k1);
        order(k2, k3);
        order(k0, k2);
        order(k1, k3);
        order(k1, k2);
        auto child = [&](uint32_t k) {
          const uint32_t a = (k & 1u) ? ch.y : ch.x, b = (k & 1u) ? ch.w : ch.z;
          return (k & 2u) ? b : a;
        };
        auto entry = [&](uint32_t k) { return ((uint64_t)k << 32) | child(k); };
        if (k3 != kMiss) st.push(sp++, entry(k3));
        if (k2 != kMiss) st.push(sp++, entry(k2));
        if (k1 != kMiss) st.push(sp++, entry(k1));
        return k0 != kMiss ? child(k0) : pop();
      } else {
        // the last child entered is next, the ones before it are stacked; with
        // room for three more in LDS in every lane, without a look at each
        const bool p0 = h0 && (h1 || h2 || h3), p1 = h1 && (h2 || h3), p2 = h2 && h3;
        const uint32_t next = h3 ? ch.w : h2 ? ch.z : h1 ? ch.y : ch.x;
        if (__ballot(sp > S - 3) == 0) {
          if (p0) st.e[64 * sp++] = ch.x;
          if (p1) st.e[64 * sp++] = ch.y;
          if (p2) st.e[64 * sp++] = ch.z;
        } else {
          if (p0) st.push(sp++, ch.x);
          if (p1) st.push(sp++, ch.y);
          if (p2) st.push(sp++, ch.z);
        }
        return h0 || h1 || h2 || h3 ? next : pop();
      }
    };
    float t[4];
    bool h[4];
    auto box = [&](int k, float xn, float xf, float yn, float yf, float zn, float zf) {
      t[k] = fmaxf(fmaxf(xn, yn), fmaxf(zn, tmin));
      h[k] = t[k] <= fminf(fminf(xf, yf), fminf(zf, tbest));
    };
    auto boxes = [&](const Planes &n) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        box(k, __builtin_fmaf(n.ax[k], ix, nx), __builtin_fmaf(n.bx[k], ix, fx),
            __builtin_fmaf(n.ay[k], iy, ny), __builtin_fmaf(n.by[k], iy, fy),
            __builtin_fmaf(n.az[k], iz, nz), __builtin_fmaf(n.bz[k], iz, fz));
    };
    // lanes of several octants (nx == fx and so on): each takes the nearer
    // plane's time per axis; a missing child's planes are swapped, so that its
    // box would be all of space
    auto boxes_mixed = [&](const Planes &n) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float xa = __builtin_fmaf(n.ax[k], ix, nx), xb = __builtin_fmaf(n.bx[k], ix, nx),
                    ya = __builtin_fmaf(n.ay[k], iy, ny), yb = __builtin_fmaf(n.by[k], iy, ny),
                    za = __builtin_fmaf(n.az[k], iz, nz), zb = __builtin_fmaf(n.bz[k], iz, nz);
        box(k, fminf(xa, xb), fmaxf(xa, xb), fminf(ya, yb), fmaxf(ya, yb), fminf(za, zb),
            fmaxf(za, zb));
        h[k] = h[k] && n.ch[k] != kBvhLeaf;
      }
    };
    for (;;) {
      while (!(cur & kBvhLeaf)) {
        Planes n;
        const uint32_t u = (uint32_t)__builtin_amdgcn_readfirstlane((int)cur);
        if (uni && __ballot(cur != u) == 0) {
          const auto *q = (const __attribute__((address_space(4))) char *)(base + ((size_t)u << 7));
          const uint32_t ux = (uint32_t)__builtin_amdgcn_readfirstlane((int)sx),
                         uy = (uint32_t)__builtin_amdgcn_readfirstlane((int)sy),
                         uz = (uint32_t)__builtin_amdgcn_readfirstlane((int)sz);
          n.load(q + ux, q + (ux ^ 16u), q + 32 + uy, q + 32 + (uy ^ 16u), q + 64 + uz,
                 q + 64 + (uz ^ 16u), q + 96);
          if (__ballot(sx != ux || sy != uy || sz != uz) == 0) boxes(n);
          else boxes_mixed(n);
        } else {
          const uint32_t at = cur << 7;
          const uint32_t px = at | sx, py = at | sy, pz = at | sz;
          n.load(base + px, base + (px ^ 16u), base + py + 32, base + (py ^ 16u) + 32,
                 base + pz + 64, base + (pz ^ 16u) + 64, base + at + 96);
          boxes(n);
        }
        cur = take(h[0], h[1], h[2], h[3], t[0], t[1], t[2], t[3], n.ch);
      }
      if (cur == kDone) break;
      const uint32_t first = cur & kBvhFirstMask, cnt = (cur & ~kBvhLeaf) >> kBvhCntShift;
      for (uint32_t k = first; k < first + cnt; ++k)
        tri_test<SKIPSKY>(refs, k, ox, oy, oz, dx, dy, dz, tmin, skip, tbest, best, best_id,
                          best_ref);
      if (ANY && best != best0) return true;
      cur = pop();
      if (cur == kDone) break;
    }
    return best != best0;
  }
};

// Closest hit in [tmin, tmax).
template <class Tracer>
__device__ __forceinline__ void trace_ray(const DevScene &sc, Tracer &tr, float ox, float oy,
                                          float oz, float dx, float dy, float dz, float tmin,
                                          float tmax, int32_t skip, float &t_out,
                                          int32_t &best_out, int32_t &id_out) {
  float tbest = tmax;
  int32_t best = -1, best_id = 0;
  t_out = 0.0f;
  best_out = -1;
  id_out = 0;
  if (sc.empty) return;
  uint32_t ref = kNoRef;
  tr.begin(ox, oy, oz, dx, dy, dz);
  if (tr.template full<false, false>(tmin, skip, tbest, best, best_id, ref)) {
    t_out = tbest;
    best_out = best;
    id_out = best_id;
  }
}

// Direction and length of a segment: dir = delta * (1/len).
__device__ __forceinline__ float segment_dir(float sx, float sy, float sz, float ex, float ey,
                                             float ez, float &dx, float &dy, float &dz) {
  const float vx = ex - sx, vy = ey - sy, vz = ez - sz;
  const float len2 = (vx * vx + vy * vy) + vz * vz;
  const float len = __builtin_sqrtf(len2);
  const float inv = 1.0f / len;
  dx = vx * inv;
  dy = vy * inv;
  dz = vz * inv;
  return len;
}

// TestLineDoesHitSky for one segment (raytracer/trace/testline.go:22-51):
// dir = delta * (1/len), trace [0, len), occluded iff the closest hit is not
// a TRACE_ID_SKY triangle.  Returns visible; *sky = closest hit is sky.
// With sky triangles present this is evaluated in two walks with the same
// result: the closest sky hit (ts, is) on the sky-only tree, then the full
// tree stops at the first non-sky hit before (ts, is) in (t, index) order;
// the segment is occluded iff there is one.
//
// occluder (in/out): a record of the full tree to test first (kNoRef
// for none), typically the triangle that blocked the caller's previous,
// nearby segment.  It is tested with the same arithmetic and bound as the
// walk, so a hit there is exactly a hit the walk would accept and the result
// does not depend on it.  On return it holds the blocking triangle found, if
// any, else it is unchanged.
template <class Tracer>
__device__ __forceinline__ bool test_line_cached(const DevScene &sc, Tracer &tr, float sx,
                                                 float sy, float sz, float ex, float ey, float ez,
                                                 int32_t skip, bool &sky, uint32_t &occluder) {
  float dx, dy, dz;
  const float len = segment_dir(sx, sy, sz, ex, ey, ez, dx, dy, dz);
  sky = false;
  if (sc.empty) return true;
  float t = len;
  int32_t best = -1, id = 0;
  uint32_t ref = kNoRef;
  tr.begin(sx, sy, sz, dx, dy, dz);
  if (sc.has_sky) tr.template sky<false>(0.0f, skip, t, best, id, ref);
  const int32_t sky_best = best;
  bool occluded = false;
  if (occluder != kNoRef) {
    tri_test<true>(sc.bvh_refs, occluder, sx, sy, sz, dx, dy, dz, 0.0f, skip, t, best, id, ref);
    occluded = best != sky_best;
  }
  if (!occluded) {
    ref = kNoRef;
    occluded = tr.template full<true, true>(0.0f, skip, t, best, id, ref);
    if (occluded) occluder = ref;
  }
  sky = !occluded && sky_best >= 0;
  return !occluded;
}
// TestLineDoesHitSky without an occluder hint, with the walks in the order
// that suits a visible segment: any opaque hit on [0, len) first.  Without
// one the segment is visible, and its closest hit is sky iff the sky tree
// has any hit on [0, len).  With one, the closest sky hit before it in
// (t, index) order (none: occluded), then any opaque hit before that sky
// hit (test_line_cached's second walk) decide; a sky hit found that way is
// the closest of all, since every sky hit it passed over lies after an
// opaque one.  Same results as test_line_cached.
template <class Tracer>
__device__ __forceinline__ bool test_line(const DevScene &sc, Tracer &tr, float sx, float sy,
                                          float sz, float ex, float ey, float ez, int32_t skip,
                                          bool &sky) {
  float dx, dy, dz;
  const float len = segment_dir(sx, sy, sz, ex, ey, ez, dx, dy, dz);
  sky = false;
  if (sc.empty) return true;
  float t = len;
  int32_t best = -1, id = 0;
  uint32_t ref = kNoRef;
  tr.begin(sx, sy, sz, dx, dy, dz);
  for (int pass = 0;; ++pass) {  // one copy of the walk's code
    if (!tr.template full<true, true>(0.0f, skip, t, best, id, ref)) {
      sky = pass != 0 ||
            (sc.has_sky && tr.template sky<false>(0.0f, skip, t, best, id, ref));
      return true;
    }
    if (pass != 0 || !sc.has_sky || !tr.template sky<false>(0.0f, skip, t, best, id, ref))
      return false;
  }
}

// test_line's visibility without its sky output, with the walks in the
// order that suits a visible segment: first any non-sky hit on [0, len)
// (none: visible, and the sky tree is never walked); then the closest sky
// hit before that one in (t, index) order (none: the closest hit is not
// sky, occluded); then, as test_line does, any non-sky hit before that sky
// hit.  The three steps decide what test_line decides: a sky hit found in
// the second is the closest of all, since every sky hit it passed over lies
// after a non-sky hit.
template <class Tracer>
__device__ __forceinline__ bool segment_visible(const DevScene &sc, Tracer &tr, float sx, float sy,
                                                float sz, float ex, float ey, float ez,
                                                int32_t skip) {
  float dx, dy, dz;
  const float len = segment_dir(sx, sy, sz, ex, ey, ez, dx, dy, dz);
  if (sc.empty) return true;
  float t = len;
  int32_t best = -1, id = 0;
  uint32_t ref = kNoRef;
  tr.begin(sx, sy, sz, dx, dy, dz);
  for (int pass = 0;; ++pass) {  // one copy of the walk's code
    if (!tr.template full<true, true>(0.0f, skip, t, best, id, ref)) return true;
    if (pass != 0 || !sc.has_sky || !tr.template sky<false>(0.0f, skip, t, best, id, ref))
      return false;
  }
}

// The first half of test_line_cached alone: whether the segment is occluded
// by `occluder` (a record of the full tree) as test_line would decide it
// (the closest sky hit first, then the same hit test and bound).  False
// means only that this triangle does not decide it.
template <class Tracer>
__device__ __forceinline__ bool occluded_by(const DevScene &sc, Tracer &tr, float sx, float sy,
                                            float sz, float ex, float ey, float ez, int32_t skip,
                                            uint32_t occluder) {
  float dx, dy, dz;
  const float len = segment_dir(sx, sy, sz, ex, ey, ez, dx, dy, dz);
  if (sc.empty) return false;
  float t = len;
  int32_t best = -1, id = 0;
  uint32_t ref = kNoRef;
  if (sc.has_sky) {
    tr.begin(sx, sy, sz, dx, dy, dz);
    tr.template sky<false>(0.0f, skip, t, best, id, ref);
  }
  const int32_t sky_best = best;
  tri_test<true>(sc.bvh_refs, occluder, sx, sy, sz, dx, dy, dz, 0.0f, skip, t, best, id, ref);
  return best != sky_best;
}

}  // namespace vr
