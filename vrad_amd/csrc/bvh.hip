// Device builder of the 4-wide bounding-volume hierarchy the visibility
// kernels walk (trace_dev.h::BvhTracer).  Results do not depend on the tree:
// a walk returns the first hit in (t, triangle) order among all triangles, as
// long as every box holds every point at which the triangle test can accept a
// hit.  The kd-tree stays for the plain path, for scenes past the hierarchy's
// node limit and for vr_scene_get_kdtree.
//
//  k_bvh_bounds   per triangle, the box of its acceptance region (below)
//  k_bvh_first    first position of each triangle in the kd-tree's index
//  k_bvh_flag /   list: its leaves in depth-first order are a spatial order,
//  k_bvh_order    so no sort is needed
//  k_ploc_nn /    bottom-up clustering (after Meister and Bittner, "Parallel
//  k_ploc_merge   Locally-Ordered Clustering for Bounding Volume Hierarchy
//  k_ploc_final   Construction", IEEE TVCG 2018): every cluster looks kPlocR
//                 places to either side for the neighbour whose union box has
//                 the least area, mutual choices merge, the rest is compacted;
//                 two launches per round, the last 2048 clusters in one
//                 workgroup (k_ploc_final)
//  k_bvh_collapse binary tree to 4-wide nodes, level by level from the root,
//                 opening the child with the largest area first
//
// Why this tree: counted on the CPU over an 8x8-room level (179,506
// triangles), a wave of 64 MakeTransfers segments takes 14-18 node steps of
// the 4-wide tree and 1-2 triangle tests where the kd-tree took 60-140 steps
// and 40-110 tests: its cells straddle the walls, so a segment that runs
// along one tests every triangle it passes, while the boxes of a wall's
// triangles are flat and a segment 0.1 above misses them.  Clustering in kd
// order came within 5 % of a binned SAH build from the top (13.5 / 14.6 /
// 17.6 / 21.6 against 13.8 / 17.8 / 19.9 / 23.0 steps on four batches) and
// needs no sort; splitting by Morton code took 19.4 / 19.9 / 27.9 / 27.5.
#include <algorithm>
#include <string>
#include <vector>

#include "kernels.h"
#include "vr_internal.h"

namespace vr {
namespace {

constexpr int kPlocR = 8;        // neighbours looked at to either side
constexpr int kPlocB = 256;      // clusters per workgroup of a round
constexpr int kPlocFinal = 2048; // clusters the last workgroup takes over
constexpr int kLeafTris = 2;     // triangles per leaf: a quad's two share a box
constexpr int kMaxLevels = kBvhStack / 3;

struct Box {
  float mn[3], mx[3];
};
struct Node2 {  // binary node: leaves 0 .. m - 1 (in order), then merges
  Box b;
  int32_t l, r;   // children (-1: a leaf, whose triangle is order[index])
  int32_t cnt;    // triangles below
};
// counters of one build
struct PlocState {
  int32_t n;      // clusters
  int32_t nodes;  // binary nodes so far
};

__device__ __forceinline__ Box box_union(const Box &a, const Box &b) {
  Box r;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    r.mn[c] = fminf(a.mn[c], b.mn[c]);
    r.mx[c] = fmaxf(a.mx[c], b.mx[c]);
  }
  return r;
}
__device__ __forceinline__ float box_area(const Box &b) {
  const float x = b.mx[0] - b.mn[0], y = b.mx[1] - b.mn[1], z = b.mx[2] - b.mn[2];
  return x * y + y * z + z * x;
}

// The box of every point p = o + t d at which tri_test can accept a hit at
// the t it computes, for origins with |o| <= M (M: the scene's largest
// coordinate; farther origins widen the walk's slabs instead, BvhTracer::begin).
// With u = 2^-24:
//  - The test accepts when the rounded b0 = E0 h0 + E1 h1 + E2 >= 0, b1 >= 0
//    and b0 + b1 <= 1.  For |h| <= 2M the rounding of b0 is at most
//    e0 = 4u ((|E0| + |E1|) 2M + |E2|), so (h0, h1) lies in the triangle
//    b0 >= -e0, b1 >= -e1, b0 + b1 <= 1 + u + e0 + e1 of the stored edge
//    equations, whose corners are taken in FP64.  For a sliver that region is
//    much longer than the triangle; one that leaves |h| <= 2M gets a box that
//    is always entered.
//  - h differs from p's two coordinates by at most 2u (4M + |o|), and p lies
//    off the plane N p = D by the rounding of t, at most 24u (M + |o|) along
//    the dropped axis (|N_drop| >= 1/sqrt 3), plus the first difference at
//    slope <= 1 per axis: 68uM in all for |o| <= M.
//  - The slab arithmetic of the walk is off by less than 8uM.
// The corners' box is widened by 96uM per side.  A triangle whose normal holds
// a NaN never passes the test and is left out (flag 0).
__global__ __launch_bounds__(256) void k_bvh_bounds(const float4 *__restrict__ tris, int64_t n,
                                                    float M, Box *__restrict__ box,
                                                    uint8_t *__restrict__ live,
                                                    uint32_t *__restrict__ first) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  first[i] = 0xffffffffu;  // in no leaf (k_bvh_first)
  const float4 q0 = tris[3 * i], q1 = tris[3 * i + 1], q2 = tris[3 * i + 2];
  const float N[3] = {q0.x, q0.y, q0.z};
  Box b;
  live[i] = !(N[0] != N[0] || N[1] != N[1] || N[2] != N[2]);
  const uint32_t cs = __float_as_uint(q2.w);
  const int c0 = (int)(cs & 255u) % 3, c1 = (int)((cs >> 8) & 255u) % 3, cd = 3 - c0 - c1;
  const double E0 = q1.y, E1 = q1.z, E2 = q1.w, E3 = q2.x, E4 = q2.y, E5 = q2.z;
  const double u = 0x1p-24, H = 2.0 * M;
  const double e0 = 4.0 * u * ((fabs(E0) + fabs(E1)) * H + fabs(E2));
  const double e1 = 4.0 * u * ((fabs(E3) + fabs(E4)) * H + fabs(E5));
  const double top = 1.0 + u + e0 + e1;
  const double det = E0 * E4 - E1 * E3;
  bool ok = c0 != c1 && fabs(det) > 0x1p-40 * (fabs(E0 * E4) + fabs(E1 * E3)) &&
            fabs((double)N[cd < 0 || cd > 2 ? 0 : cd]) > 0.5 && q0.w == q0.w;
  double mn[3] = {1e300, 1e300, 1e300}, mx[3] = {-1e300, -1e300, -1e300};
  const double r[3][2] = {{-e0, -e1}, {top + e1, -e1}, {-e0, top + e0}};
  for (int k = 0; ok && k < 3; ++k) {
    const double a = r[k][0] - E2, c = r[k][1] - E5;
    double p[3] = {0.0, 0.0, 0.0};
    p[c0] = (a * E4 - E1 * c) / det;
    p[c1] = (E0 * c - a * E3) / det;
    ok = fabs(p[c0]) <= H && fabs(p[c1]) <= H;  // false for NaN
    p[cd] = (((double)q0.w - (double)N[c0] * p[c0]) - (double)N[c1] * p[c1]) / (double)N[cd];
    ok = ok && fabs(p[cd]) <= 8.0 * M;
    for (int q = 0; q < 3; ++q) {
      mn[q] = fmin(mn[q], p[q]);
      mx[q] = fmax(mx[q], p[q]);
    }
  }
  const double e = 96.0 * u * M;
  for (int q = 0; q < 3; ++q) {
    b.mn[q] = ok ? (float)(mn[q] - e) : -3e38f;
    b.mx[q] = ok ? (float)(mx[q] + e) : 3e38f;
  }
  box[i] = b;
}

__global__ __launch_bounds__(256) void k_bvh_first(const int32_t *__restrict__ idx, int64_t n_idx,
                                                   uint32_t *__restrict__ first) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k < n_idx) atomicMin(&first[idx[k]], (uint32_t)k);
}

// Position k of the order's source: the index list, then (all) every triangle
// that is not in the list.
__device__ __forceinline__ bool order_take(const int32_t *idx, int64_t n_idx, int64_t n_all,
                                           const uint32_t *first, const uint8_t *live, int64_t k,
                                           int32_t &tri) {
  if (k >= n_idx + n_all) return false;
  tri = k < n_idx ? idx[k] : (int32_t)(k - n_idx);
  return live[tri] && first[tri] == (k < n_idx ? (uint32_t)k : 0xffffffffu);
}

// taken entries per 1024 source positions
__global__ __launch_bounds__(1024) void k_bvh_flag(const int32_t *__restrict__ idx, int64_t n_idx,
                                                   int64_t n_all,
                                                   const uint32_t *__restrict__ first,
                                                   const uint8_t *__restrict__ live,
                                                   int32_t *__restrict__ cnt) {
  int32_t tri;
  const bool t = order_take(idx, n_idx, n_all, first, live,
                            (int64_t)blockIdx.x * 1024 + threadIdx.x, tri);
  const int c = __syncthreads_count(t);
  if (threadIdx.x == 0) cnt[blockIdx.x] = c;
}

// exclusive prefix of one value per thread over a workgroup of B threads
template <int B>
__device__ __forceinline__ int wg_scan(int v, int *s_w, int &total) {
  const int lane = (int)(threadIdx.x & 63), w = (int)(threadIdx.x >> 6);
  int x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  if (lane == 63) s_w[w] = x;
  __syncthreads();
  int base = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < B / 64; ++k) {
    base += k < w ? s_w[k] : 0;
    tot += s_w[k];
  }
  __syncthreads();
  total = tot;
  return base + x - v;
}

// sum over v[0, n) with the whole workgroup of B threads (every thread gets it)
template <int B>
__device__ __forceinline__ int wg_sum(const int32_t *v, int n, int stride, int *s_w) {
  int x = 0;
  for (int k = (int)threadIdx.x; k < n; k += B) x += v[(int64_t)k * stride];
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d);
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = x;
  __syncthreads();
  int t = 0;
#pragma unroll
  for (int k = 0; k < B / 64; ++k) t += s_w[k];
  __syncthreads();
  return t;
}

// The leaves in order: binary nodes 0 .. m - 1 and the first clusters.
__global__ __launch_bounds__(1024) void k_bvh_order(
    const int32_t *__restrict__ idx, int64_t n_idx, int64_t n_all,
    const uint32_t *__restrict__ first, const uint8_t *__restrict__ live,
    const int32_t *__restrict__ cnt, const Box *__restrict__ box, int32_t *__restrict__ order,
    Node2 *__restrict__ nodes, Box *__restrict__ cbox, int32_t *__restrict__ cid,
    PlocState *__restrict__ st) {
  __shared__ int s_w[16];
  const int base = wg_sum<1024>(cnt, (int)blockIdx.x, 1, s_w);
  int32_t tri = 0;
  const bool t = order_take(idx, n_idx, n_all, first, live,
                            (int64_t)blockIdx.x * 1024 + threadIdx.x, tri);
  int total;
  const int at = base + wg_scan<1024>(t ? 1 : 0, s_w, total);
  if (t) {
    const Box b = box[tri];
    order[at] = tri;
    nodes[at] = Node2{b, -1, -1, 1};
    cbox[at] = b;
    cid[at] = at;
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *st = PlocState{base + total, base + total};
}

// Choice of cluster i (box a) among the R clusters to either side: least area
// of the union, ties to the least i ^ j.  That key is the same seen from
// either side and unique per i, so the least pair of all is always mutual and
// every round merges at least it.  `pair`: i ^ 1 outright (the balanced tree).
template <class GET>
__device__ __forceinline__ int ploc_choice(int i, int n, bool pair, const GET &get) {
  if (pair) return (i ^ 1) < n ? (i ^ 1) : i;
  const Box a = get(i);
  uint64_t best = ~0ull;
  int bj = i;
  for (int j = max(0, i - kPlocR); j <= min(n - 1, i + kPlocR); ++j) {
    if (j == i) continue;
    const float ar = box_area(box_union(a, get(j)));
    const uint64_t key = ((uint64_t)__float_as_uint(fminf(ar, 3e38f)) << 32) | (uint32_t)(i ^ j);
    if (key < best) {
      best = key;
      bj = j;
    }
  }
  return bj;
}

// A round's choices: own clusters and kPlocR to either side (so that a
// workgroup knows its own survivors); counts per workgroup: survivors, merges.
__global__ __launch_bounds__(kPlocB) void k_ploc_nn(const PlocState *__restrict__ st, int pair,
                                                    const Box *__restrict__ cbox,
                                                    int32_t *__restrict__ choice,
                                                    int32_t *__restrict__ cnt) {
  constexpr int R = kPlocR, W = kPlocB + 4 * R;
  __shared__ Box s_b[W];
  __shared__ int s_c[kPlocB + 2 * R];
  __shared__ int s_w[kPlocB / 64];
  const int n = st->n, b0 = (int)blockIdx.x * kPlocB;
  if (b0 >= n || n <= 1) return;
  for (int k = (int)threadIdx.x; k < W; k += kPlocB) {
    const int i = b0 - 2 * R + k;
    if (i >= 0 && i < n) s_b[k] = cbox[i];
  }
  __syncthreads();
  auto get = [&](int i) -> const Box & { return s_b[i - b0 + 2 * R]; };
  for (int k = (int)threadIdx.x; k < kPlocB + 2 * R; k += kPlocB) {
    const int i = b0 - R + k;
    s_c[k] = i >= 0 && i < n ? ploc_choice(i, n, pair != 0, get) : -1;
  }
  __syncthreads();
  const int i = b0 + (int)threadIdx.x;
  int surv = 0, lead = 0;
  if (i < n) {
    const int j = s_c[i - b0 + R];
    const bool mutual = j != i && s_c[j - b0 + R] == i;
    surv = !(mutual && i > j);
    lead = mutual && i < j;
    choice[i] = mutual ? j : i;
  }
  int ts, tl;
  (void)wg_scan<kPlocB>(surv, s_w, ts);
  (void)wg_scan<kPlocB>(lead, s_w, tl);
  if (threadIdx.x == 0) {
    cnt[2 * blockIdx.x] = ts;
    cnt[2 * blockIdx.x + 1] = tl;
  }
}

__global__ __launch_bounds__(kPlocB) void k_ploc_merge(
    const PlocState *__restrict__ st, PlocState *__restrict__ next, const Box *__restrict__ cbox,
    const int32_t *__restrict__ cid, const int32_t *__restrict__ choice,
    const int32_t *__restrict__ cnt, Box *__restrict__ nbox, int32_t *__restrict__ nid,
    Node2 *__restrict__ nodes) {
  __shared__ int s_w[kPlocB / 64];
  const PlocState s = *st;
  const int b0 = (int)blockIdx.x * kPlocB;
  if (s.n <= 1) {  // done: carry the state and the root on
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      *next = s;
      if (s.n == 1) {
        nbox[0] = cbox[0];
        nid[0] = cid[0];
      }
    }
    return;
  }
  if (b0 >= s.n) return;
  const int sb = wg_sum<kPlocB>(cnt, (int)blockIdx.x, 2, s_w);
  const int lb = wg_sum<kPlocB>(cnt + 1, (int)blockIdx.x, 2, s_w);
  const int i = b0 + (int)threadIdx.x;
  int j = i, surv = 0, lead = 0;
  if (i < s.n) {
    j = choice[i];
    surv = j >= i;
    lead = j > i;
  }
  int ts, tl;
  const int at = sb + wg_scan<kPlocB>(surv, s_w, ts);
  const int ln = lb + wg_scan<kPlocB>(lead, s_w, tl);
  if (lead) {
    const int32_t l = cid[i], r = cid[j];
    const Box b = box_union(cbox[i], cbox[j]);
    const int32_t id = s.nodes + ln;
    nodes[id] = Node2{b, l, r, nodes[l].cnt + nodes[r].cnt};
    nbox[at] = b;
    nid[at] = id;
  } else if (surv) {
    nbox[at] = cbox[i];
    nid[at] = cid[i];
  }
  if (b0 + kPlocB >= s.n && threadIdx.x == 0)
    *next = PlocState{sb + ts, s.nodes + lb + tl};
}

// The last rounds in one workgroup; *root = the root's binary node.  Also
// starts the collapse's counters lv[0, 128): one node in level 0 (none without
// triangles).
__global__ __launch_bounds__(1024) void k_ploc_final(const PlocState *__restrict__ st, int pair,
                                                     const Box *__restrict__ cbox,
                                                     const int32_t *__restrict__ cid,
                                                     Node2 *__restrict__ nodes,
                                                     int32_t *__restrict__ root,
                                                     int32_t *__restrict__ lv) {
  constexpr int PER = kPlocFinal / 1024;
  __shared__ Box s_b[kPlocFinal];
  __shared__ int32_t s_id[kPlocFinal];
  __shared__ int16_t s_c[kPlocFinal];
  __shared__ int s_w[16];
  int n = min(st->n, kPlocFinal), base = st->nodes;
  const int t = (int)threadIdx.x;
  if (t < 128) lv[t] = t == 0 && n > 0 ? 1 : 0;
  for (int k = t; k < n; k += 1024) {
    s_b[k] = cbox[k];
    s_id[k] = cid[k];
  }
  __syncthreads();
  auto get = [&](int i) -> const Box & { return s_b[i]; };
  // a round at least merges one pair; past 64 rounds neighbours are paired
  // outright, so the loop ends after at most 64 + log2(2048) rounds
  for (int round = 0; n > 1; ++round) {
    const bool pr = pair != 0 || round >= 64;
    for (int k = t; k < n; k += 1024) s_c[k] = (int16_t)ploc_choice(k, n, pr, get);
    __syncthreads();
    Box b[PER];
    int32_t id[PER];
    int surv = 0, lead = 0, kind[PER];  // 0 gone, 1 kept, 2 merged
    int other[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int i = PER * t + q;
      kind[q] = 0;
      other[q] = i;
      if (i < n) {
        const int j = s_c[i];
        const bool mutual = j != i && s_c[j] == i;
        kind[q] = mutual ? (i < j ? 2 : 0) : 1;
        other[q] = j;
        b[q] = s_b[i];
        id[q] = s_id[i];
        surv += kind[q] != 0;
        lead += kind[q] == 2;
      }
    }
    int ts, tl;
    int at = wg_scan<1024>(surv, s_w, ts);
    int ln = wg_scan<1024>(lead, s_w, tl);
#pragma unroll
    for (int q = 0; q < PER; ++q)
      if (kind[q] == 2) {
        const int32_t l = id[q], r = s_id[other[q]];
        b[q] = box_union(b[q], s_b[other[q]]);
        id[q] = base + ln++;
        nodes[id[q]] = Node2{b[q], l, r, nodes[l].cnt + nodes[r].cnt};
      }
    __syncthreads();  // every read of s_b / s_id is done (and the nodes written)
#pragma unroll
    for (int q = 0; q < PER; ++q)
      if (kind[q]) {
        s_b[at] = b[q];
        s_id[at++] = id[q];
      }
    n = ts;
    base += tl;
    __syncthreads();
  }
  if (t == 0 && n > 0) *root = s_id[0];
}

// One level of the 4-wide tree: wide node w (the queue position of its binary
// root) takes the binary children, opening the inner one of the largest area
// until there are four (`even`: both children once, two binary levels per wide
// level, which bounds the depth).  Subtrees of at most kLeafTris triangles
// become leaves, whose records are written next to their siblings'.  Children
// are queued next to each other for the next level.
// The level's nodes are queue[begin, begin + n); next: nodes of the next level
// so far; tri_cnt: leaf records so far.
template <int B>
__device__ __forceinline__ void collapse_level(
    const Node2 *__restrict__ nodes, const int32_t *__restrict__ order,
    const float4 *__restrict__ tris, int begin, int n, int even, int32_t *next, int32_t *tri_cnt,
    int32_t *__restrict__ queue, int64_t cap, float4 *__restrict__ wide,
    float4 *__restrict__ refs) {
  __shared__ int s_w[B / 64];
  __shared__ int s_q, s_t;
  for (int b0 = (int)blockIdx.x * B; b0 < n; b0 += (int)gridDim.x * B) {
    const int i = b0 + (int)threadIdx.x;
    int32_t c[4] = {-1, -1, -1, -1};
    int nc = 0, inner = 0, nt = 0;
    if (i < n) {
      const int32_t r = queue[begin + i];
      c[0] = r;
      nc = 1;
      // open: entries with more than kLeafTris triangles
      auto open = [&](int k) {
        const Node2 &nd = nodes[c[k]];
        c[nc++] = nd.r;
        c[k] = nd.l;
      };
      if (nodes[r].cnt > kLeafTris) open(0);
      if (even) {
        const int two = nc;
        for (int k = 0; k < two; ++k)
          if (nodes[c[k]].cnt > kLeafTris) open(k);
      } else {
        while (nc < 4) {
          int best = -1;
          float ba = -1.0f;
          for (int k = 0; k < nc; ++k) {
            const Node2 &nd = nodes[c[k]];
            const float ar = box_area(nd.b);
            if (nd.cnt > kLeafTris && !(ar <= ba)) {
              best = k;
              ba = ar;
            }
          }
          if (best < 0) break;
          open(best);
        }
      }
      for (int k = 0; k < nc; ++k) {
        const int32_t m = nodes[c[k]].cnt;
        if (m > kLeafTris) ++inner;
        else nt += m;
      }
    }
    int ti, tt;
    const int qi = wg_scan<B>(inner, s_w, ti);
    const int qt = wg_scan<B>(nt, s_w, tt);
    if (threadIdx.x == 0) {
      s_q = ti ? atomicAdd(next, ti) : 0;
      s_t = tt ? atomicAdd(tri_cnt, tt) : 0;
    }
    __syncthreads();
    int at = begin + n + s_q + qi, tr = s_t + qt;
    __syncthreads();
    if (i < n) {
      // children planes by axis: (min, max) of x, y, z, four children each
      float v[6][4];
      uint32_t ch[4];
      for (int k = 0; k < 4; ++k) {
        if (k >= nc) {  // no child: a box no ray enters, and a leaf of none
          for (int a = 0; a < 3; ++a) {
            v[2 * a][k] = 3e38f;
            v[2 * a + 1][k] = -3e38f;
          }
          ch[k] = kBvhLeaf;
          continue;
        }
        const Node2 &nd = nodes[c[k]];
        for (int a = 0; a < 3; ++a) {
          v[2 * a][k] = nd.b.mn[a];
          v[2 * a + 1][k] = nd.b.mx[a];
        }
        if (nd.cnt > kLeafTris) {
          if (at < cap) queue[at] = c[k];
          ch[k] = (uint32_t)at++;
          continue;
        }
        ch[k] = kBvhLeaf | ((uint32_t)nd.cnt << kBvhCntShift) | (uint32_t)tr;
        int32_t leaf[kLeafTris] = {c[k], -1};
        if (nd.l >= 0) {
          leaf[0] = nd.l;
          leaf[1] = nd.r;
        }
        for (int q = 0; q < nd.cnt; ++q, ++tr) {
          const int32_t ti2 = order[leaf[q]];
          const float4 t0 = tris[3 * (int64_t)ti2], t1 = tris[3 * (int64_t)ti2 + 1],
                       t2 = tris[3 * (int64_t)ti2 + 2];
          const uint32_t cs = __float_as_uint(t2.w);
          const uint32_t meta = (uint32_t)ti2 | ((cs & 3u) << 28) | (((cs >> 8) & 3u) << 30);
          refs[3 * (int64_t)tr] = t0;
          refs[3 * (int64_t)tr + 1] = make_float4(t1.y, t1.z, t1.w, t2.x);
          refs[3 * (int64_t)tr + 2] = make_float4(t2.y, t2.z, t1.x, __uint_as_float(meta));
        }
      }
      float4 *o = wide + 8 * (int64_t)(begin + i);
      for (int a = 0; a < 6; ++a) o[a] = make_float4(v[a][0], v[a][1], v[a][2], v[a][3]);
      o[6] = make_float4(__uint_as_float(ch[0]), __uint_as_float(ch[1]), __uint_as_float(ch[2]),
                         __uint_as_float(ch[3]));
      o[7] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
  }
}

// cnt[l]: nodes of level l
__global__ __launch_bounds__(256) void k_bvh_collapse(
    const Node2 *__restrict__ nodes, const int32_t *__restrict__ order,
    const float4 *__restrict__ tris, int level, int even, int32_t *__restrict__ cnt,
    int32_t *__restrict__ tri_cnt, int32_t *__restrict__ queue, int64_t cap,
    float4 *__restrict__ wide, float4 *__restrict__ refs) {
  int begin = 0;
  for (int l = 0; l < level; ++l) begin += cnt[l];
  collapse_level<256>(nodes, order, tris, begin, cnt[level], even, &cnt[level + 1], tri_cnt, queue,
                      cap, wide, refs);
}

// All levels in one workgroup, for the trees that one workgroup clusters: a
// launch per level was 12 launches of some 5 us, 78 us for 1,584 triangles
// against 45.  With the small scenes' records written in place, one upload per
// tree and their counts read into pinned memory, the build of 96 triangles went
// from 235 to 172 us and that of 1,584 from 1.82 to 1.66 ms (86 us and 1.55 ms
// without the hierarchy).
__global__ __launch_bounds__(1024) void k_bvh_collapse_all(
    const Node2 *__restrict__ nodes, const int32_t *__restrict__ order,
    const float4 *__restrict__ tris, int even, int32_t *__restrict__ cnt,
    int32_t *__restrict__ tri_cnt, int32_t *__restrict__ queue, int64_t cap,
    float4 *__restrict__ wide, float4 *__restrict__ refs) {
  __shared__ int32_t s_next, s_tri;
  int begin = 0, n = cnt[0];
  if (threadIdx.x == 0) s_tri = 0;
  for (int level = 0; n > 0 && level < 126; ++level) {
    if (threadIdx.x == 0) s_next = 0;
    __syncthreads();
    collapse_level<1024>(nodes, order, tris, begin, n, even, &s_next, &s_tri, queue, cap, wide,
                         refs);
    __syncthreads();  // the next level's queue is written
    begin += n;
    n = s_next;
    if (threadIdx.x == 0) cnt[level + 1] = n;
    __syncthreads();  // and its count read, before it is cleared
  }
  if (threadIdx.x == 0) *tri_cnt = s_tri;
}

// kd-tree records of the plain path from the tree's arrays and the triangle
// records: node pairs, and 3 float4 per leaf reference (map: the tree's own
// triangle numbering, nullable)
__global__ __launch_bounds__(256) void k_kd_nodes(const uint32_t *__restrict__ children,
                                                  const uint32_t *__restrict__ split, int64_t n,
                                                  uint2 *__restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k < n) out[k] = make_uint2(children[k], split[k]);
}
__global__ __launch_bounds__(256) void k_kd_refs(const int32_t *__restrict__ idx, int64_t n,
                                                 const int32_t *__restrict__ map,
                                                 const float4 *__restrict__ tris,
                                                 float4 *__restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  const int64_t ti = map ? map[idx[k]] : idx[k];
  const float4 t0 = tris[3 * ti], t1 = tris[3 * ti + 1], t2 = tris[3 * ti + 2];
  const uint32_t cs = __float_as_uint(t2.w);
  const uint32_t meta = (uint32_t)ti | ((cs & 3u) << 28) | (((cs >> 8) & 3u) << 30);
  out[3 * k] = t0;
  out[3 * k + 1] = make_float4(t1.y, t1.z, t1.w, t2.x);
  out[3 * k + 2] = make_float4(t2.y, t2.z, t1.x, __uint_as_float(meta));
}
__global__ __launch_bounds__(256) void k_planes(const float4 *__restrict__ tris, int64_t n,
                                                float4 *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = tris[3 * i];
}

unsigned blocks_of(int64_t n, int b) { return (unsigned)std::max<int64_t>(1, (n + b - 1) / b); }

#define BVH_HIP(call)                                                                  \
  do {                                                                                 \
    const hipError_t e_ = (call);                                                      \
    if (e_ != hipSuccess) {                                                            \
      (void)hipStreamSynchronize(st);                                                  \
      return fail(e_ == hipErrorOutOfMemory ? VR_E_NOMEM : VR_E_HIP,                   \
                  std::string("BVH build: ") + #call + ": " + hipGetErrorString(e_));  \
    }                                                                                  \
  } while (0)

}  // namespace

void launch_kd_records(const uint32_t *children, const float *split, int64_t n_nodes,
                       const int32_t *idx, int64_t n_idx, const int32_t *map, const float4 *tris,
                       uint2 *nodes, float4 *refs, hipStream_t st) {
  if (n_nodes > 0)
    hipLaunchKernelGGL(k_kd_nodes, dim3(blocks_of(n_nodes, 256)), dim3(256), 0, st, children,
                       reinterpret_cast<const uint32_t *>(split), n_nodes, nodes);
  if (n_idx > 0)
    hipLaunchKernelGGL(k_kd_refs, dim3(blocks_of(n_idx, 256)), dim3(256), 0, st, idx, n_idx, map,
                       tris, refs);
}

void launch_planes(const float4 *tris, int64_t n, float4 *planes, hipStream_t st) {
  if (n > 0)
    hipLaunchKernelGGL(k_planes, dim3(blocks_of(n, 256)), dim3(256), 0, st, tris, n, planes);
}

int build_bvh(const float4 *tris, int64_t n, const int32_t *idx, int64_t n_idx, bool all, float M,
              hipStream_t st, BvhBuild *out) {
  out->n_nodes = out->n_refs = 0;
  out->levels = 0;
  if (n <= 0 || n >= (1 << kBvhCntShift)) {
    if (n > 0) return fail(VR_E_CAPACITY, "BVH build: more than 2^28 triangles");
    return VR_OK;
  }
  const int64_t src = n_idx + (all ? n : 0);
  const int64_t cap = std::max<int64_t>(1, all ? n : n_idx);  // leaves at most
  // one temporary block, carved
  struct Temp {
    char *p = nullptr;
    ~Temp() {
      dev_free(p);
    }
  } tmp;
  size_t off = 0;
  auto carve = [&](size_t bytes) {
    const size_t at = off;
    off += (bytes + 255) & ~(size_t)255;
    return at;
  };
  const int64_t order_blocks = (src + 1023) / 1024, ploc_blocks = (cap + kPlocB - 1) / kPlocB;
  const size_t o_box = carve(sizeof(Box) * (size_t)n), o_live = carve((size_t)n);
  const size_t o_first = carve(4 * (size_t)n);
  const size_t o_cnt = carve(4 * (size_t)std::max(order_blocks, 2 * ploc_blocks));
  const size_t o_order = carve(4 * (size_t)cap), o_nodes = carve(sizeof(Node2) * 2 * (size_t)cap);
  const size_t o_cb0 = carve(sizeof(Box) * (size_t)cap), o_cb1 = carve(sizeof(Box) * (size_t)cap);
  const size_t o_ci0 = carve(4 * (size_t)cap), o_ci1 = carve(4 * (size_t)cap);
  const size_t o_choice = carve(4 * (size_t)cap), o_queue = carve(4 * (size_t)cap);
  // a tree that one workgroup collapses goes straight to its final blocks
  const bool one = cap <= kPlocFinal;
  const size_t o_wide = carve(one ? 0 : 128 * (size_t)cap), o_refs = carve(one ? 0 : 48 * (size_t)cap);
  const size_t o_state = carve(2 * sizeof(PlocState) + 4), o_lv = carve(4 * 128);
  BVH_HIP((hipError_t)dev_alloc(reinterpret_cast<void **>(&tmp.p), off));
  if (one) {
    BVH_HIP((hipError_t)dev_alloc(&out->nodes, 128 * (size_t)cap));
    BVH_HIP((hipError_t)dev_alloc(&out->refs, 48 * (size_t)cap));
  }
  auto at = [&](size_t o) { return tmp.p + o; };
  Box *box = reinterpret_cast<Box *>(at(o_box));
  uint8_t *live = reinterpret_cast<uint8_t *>(at(o_live));
  uint32_t *first = reinterpret_cast<uint32_t *>(at(o_first));
  int32_t *cnt = reinterpret_cast<int32_t *>(at(o_cnt));
  int32_t *order = reinterpret_cast<int32_t *>(at(o_order));
  Node2 *nodes = reinterpret_cast<Node2 *>(at(o_nodes));
  Box *cb[2] = {reinterpret_cast<Box *>(at(o_cb0)), reinterpret_cast<Box *>(at(o_cb1))};
  int32_t *ci[2] = {reinterpret_cast<int32_t *>(at(o_ci0)), reinterpret_cast<int32_t *>(at(o_ci1))};
  int32_t *choice = reinterpret_cast<int32_t *>(at(o_choice));
  int32_t *queue = reinterpret_cast<int32_t *>(at(o_queue));
  float4 *wide = reinterpret_cast<float4 *>(one ? out->nodes : at(o_wide));
  float4 *refs = reinterpret_cast<float4 *>(one ? out->refs : at(o_refs));
  PlocState *state = reinterpret_cast<PlocState *>(at(o_state));
  int32_t *lv = reinterpret_cast<int32_t *>(at(o_lv));  // [0, 127): nodes per level; 127: leaf records
  hipLaunchKernelGGL(k_bvh_bounds, dim3(blocks_of(n, 256)), dim3(256), 0, st, tris, n, M, box, live,
                     first);
  if (n_idx > 0)
    hipLaunchKernelGGL(k_bvh_first, dim3(blocks_of(n_idx, 256)), dim3(256), 0, st, idx, n_idx, first);
  for (int pass = 0; pass < 2; ++pass) {
    // pass 1 (rare): the clustered tree was deeper than the walk's stack
    // holds, so neighbours in kd order are paired into a balanced one
    const int pair = pass;
    if (order_blocks > 1)  // one block counts for itself
      hipLaunchKernelGGL(k_bvh_flag, dim3((unsigned)order_blocks), dim3(1024), 0, st, idx, n_idx,
                         all ? n : 0, first, live, cnt);
    hipLaunchKernelGGL(k_bvh_order, dim3((unsigned)order_blocks), dim3(1024), 0, st, idx, n_idx,
                       all ? n : 0, first, live, cnt, box, order, nodes, cb[0], ci[0], state);
    BVH_HIP(hipGetLastError());
    PlocState h{(int32_t)cap, 0};  // an upper bound until the first read
    int cur = 0;
    for (int round = 0; h.n > kPlocFinal;) {
      // five rounds between two reads of the count; past 60 rounds neighbours
      // are paired outright, so the loop ends
      const int64_t grid = (h.n + kPlocB - 1) / kPlocB;
      for (int k = 0; k < 5; ++k, ++round, cur ^= 1) {
        hipLaunchKernelGGL(k_ploc_nn, dim3((unsigned)grid), dim3(kPlocB), 0, st, state + cur,
                           pair || round >= 60, cb[cur], choice, cnt);
        hipLaunchKernelGGL(k_ploc_merge, dim3((unsigned)grid), dim3(kPlocB), 0, st, state + cur,
                           state + (cur ^ 1), cb[cur], ci[cur], choice, cnt, cb[cur ^ 1],
                           ci[cur ^ 1], nodes);
      }
      BVH_HIP(hipGetLastError());
      BVH_HIP(hipMemcpyAsync(&h, state + cur, sizeof h, hipMemcpyDeviceToHost, st));
      BVH_HIP(hipStreamSynchronize(st));
    }
    hipLaunchKernelGGL(k_ploc_final, dim3(1), dim3(1024), 0, st, state + cur, pair, cb[cur], ci[cur],
                       nodes, queue, lv);
    int32_t own[128];
    int32_t *const hl = out->host ? out->host : own;
    int level = 0;
    const unsigned cg = (unsigned)std::min<int64_t>(1024, blocks_of(cap, 512));
    if (one)
      hipLaunchKernelGGL(k_bvh_collapse_all, dim3(1), dim3(1024), 0, st, nodes, order, tris, pair,
                         lv, lv + 127, queue, cap, wide, refs);
    do {
      for (int k = 0; !one && k < 12 && level < 126; ++k, ++level)
        hipLaunchKernelGGL(k_bvh_collapse, dim3(cg), dim3(256), 0, st, nodes, order, tris, level,
                           pair, lv, lv + 127, queue, cap, wide, refs);
      BVH_HIP(hipGetLastError());
      BVH_HIP(hipMemcpyAsync(hl, lv, sizeof own, hipMemcpyDeviceToHost, st));
      BVH_HIP(hipStreamSynchronize(st));
      if (one) level = 126;
    } while (hl[level] != 0 && level < kMaxLevels);
    int levels = 0;
    int64_t total = 0;
    while (levels < 126 && hl[levels] > 0) total += hl[levels++];
    const int most = pass == 0 ? std::min(kMaxLevels, tuning().bvh_levels) : kMaxLevels;
    if (levels <= most && hl[level] == 0) {
      out->n_nodes = total;
      out->n_refs = hl[127];
      out->levels = levels;
      break;
    }
    if (pass == 1) return fail(VR_E_CAPACITY, "BVH deeper than the traversal stack");
  }
  if (out->n_nodes == 0) {  // no triangle can be hit
    dev_free(out->nodes);
    dev_free(out->refs);
    out->nodes = out->refs = nullptr;
  }
  if (one || out->n_nodes == 0) return VR_OK;
  BVH_HIP((hipError_t)dev_alloc(&out->nodes, 128 * (size_t)out->n_nodes));
  BVH_HIP((hipError_t)dev_alloc(&out->refs, 48 * (size_t)out->n_refs));
  BVH_HIP(hipMemcpyAsync(out->nodes, wide, 128 * (size_t)out->n_nodes, hipMemcpyDeviceToDevice, st));
  BVH_HIP(hipMemcpyAsync(out->refs, refs, 48 * (size_t)out->n_refs, hipMemcpyDeviceToDevice, st));
  return VR_OK;
}

}  // namespace vr
