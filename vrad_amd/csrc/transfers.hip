// MakeTransfers: patch-pair visibility and CSR construction.
//
//  1. k_pair_rows   candidate pairs that pass the facing cull, a wave per patch
//                   and run of columns; TestLine(o_i + eps n_i -> o_j + eps n_j)
//                   per survivor; visible pairs set bit (i, j) of an N x N bit
//                   matrix (N^2/8 bytes: 15 GB at 341k patches, which an MI355X
//                   holds with room to spare).  The plain path lists the pairs
//                   (k_pair_cull) and traces the list (k_pair_trace_plain).
//  2. k_bits_mirror makes the matrix symmetric.
//  3. k_row_count   popcount per row; the host pads the lengths to 8 and sums
//                   them up, k_sort_* order the rows longest first.
//  4. k_row_fill    columns in ascending order, F_ij in FP32.
//  5. k_row_norm    FP64 row sum in the bounce-kernel wave order (G = 4);
//                   rows with sum > 1 are scaled by 1/sum.
#include <algorithm>

#include "kernels.h"

namespace vr {

#define VR_PI_F 3.14159265358979323846f

// A block of 256 threads tests 256 * kCullIt candidates (row, j) of one row;
// the waves keep their ballots, the block reserves its survivors' slots with
// one atomic, and every wave writes its pairs in j order.
constexpr int kCullIt = 16;

__global__ __launch_bounds__(256) void k_pair_cull(DevPatches p, int64_t np, int64_t i0,
                                                   int64_t bpr, int2 *__restrict__ pairs,
                                                   uint32_t *__restrict__ count, uint32_t cap) {
  __shared__ uint32_t s_cnt[4];
  __shared__ uint32_t s_base;
  const int64_t row = i0 + (int64_t)blockIdx.x / bpr;
  const int64_t jb = row + 1 + ((int64_t)blockIdx.x % bpr) * (256 * kCullIt);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float rx = p.ox[row], ry = p.oy[row], rz = p.oz[row];
  const float qx = p.nx[row], qy = p.ny[row], qz = p.nz[row];
  uint64_t m[kCullIt];
  uint32_t wtot = 0;
#pragma unroll
  for (int it = 0; it < kCullIt; ++it) {
    const int64_t j = jb + it * 256 + threadIdx.x;
    bool keep = false;
    if (j < np) {
      const float dx = p.ox[j] - rx, dy = p.oy[j] - ry, dz = p.oz[j] - rz;
      const float di = (qx * dx + qy * dy) + qz * dz;
      const float dj = -((p.nx[j] * dx + p.ny[j] * dy) + p.nz[j] * dz);
      keep = di > 0.0f && dj > 0.0f;
    }
    m[it] = __ballot(keep);
    wtot += (uint32_t)__popcll(m[it]);
  }
  if (lane == 0) s_cnt[wave] = wtot;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t tot = s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3];
    s_base = tot ? atomicAdd(count, tot) : 0u;
  }
  __syncthreads();
  uint32_t base = s_base;
  for (int w = 0; w < wave; ++w) base += s_cnt[w];
  const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
  for (int it = 0; it < kCullIt; ++it) {
    if ((m[it] >> lane) & 1ull) {
      const uint32_t slot = base + (uint32_t)__popcll(m[it] & below);
      if (slot < cap) pairs[slot] = make_int2((int)row, (int)(jb + it * 256 + threadIdx.x));
    }
    base += (uint32_t)__popcll(m[it]);
  }
}

void launch_pair_cull(const DevPatches &p, int64_t np, int64_t i0, int64_t i1, int2 *pairs,
                      uint32_t *count, uint32_t cap, hipStream_t st) {
  if (i1 <= i0) return;
  const int64_t maxlen = np - 1 - i0;
  if (maxlen <= 0) return;
  const int64_t bpr = (maxlen + 256 * kCullIt - 1) / (256 * kCullIt);
  hipLaunchKernelGGL(k_pair_cull, dim3((unsigned)((i1 - i0) * bpr)), dim3(256), 0, st, p, np, i0,
                     bpr, pairs, count, cap);
}

__device__ __forceinline__ void set_pair_bits(uint32_t *bits, int64_t words, int i, int j) {
  atomicOr(bits + (int64_t)i * words + (j >> 5), 1u << (j & 31));
  atomicOr(bits + (int64_t)j * words + (i >> 5), 1u << (i & 31));
}

template <int D>
__global__ __launch_bounds__(256) void k_pair_trace_plain(DevScene sc, DevPatches p,
                                                          const int2 *__restrict__ pairs,
                                                          const uint32_t *__restrict__ count,
                                                          uint32_t cap, float eps, int32_t skip,
                                                          uint32_t *__restrict__ bits,
                                                          int64_t words) {
  const uint32_t n = min(*count, cap);
  // the grid is sized for cap pairs; only the first ceil(n / 256) blocks have
  // work, and the XCD-aware remap runs over just those
  const uint32_t nb = (n + 255u) / 256u;
  if (blockIdx.x >= nb) return;
  const uint32_t k = xcd_chunk(blockIdx.x, nb) * 256 + threadIdx.x;
  if (k >= n) return;
  const int2 ij = pairs[k];
  const int i = ij.x, j = ij.y;
  ScratchStack<D> st;
  KdTracer<D> tr(sc, st);
  const bool vis = segment_visible(sc, tr, p.ox[i] + eps * p.nx[i],
                                      p.oy[i] + eps * p.ny[i], p.oz[i] + eps * p.nz[i],
                                      p.ox[j] + eps * p.nx[j], p.oy[j] + eps * p.ny[j],
                                      p.oz[j] + eps * p.nz[j], skip);
  if (vis) set_pair_bits(bits, words, i, j);
}

void launch_pair_trace(const DevScene &sc, const DevPatches &p, const int2 *pairs,
                       const uint32_t *count, uint32_t cap, float eps, int32_t skip,
                       uint32_t *bits, int64_t words, hipStream_t st) {
  if (cap == 0) return;
  hipLaunchKernelGGL(k_pair_trace_plain<kStackDepth>, dim3((cap + 255) / 256), dim3(256), 0, st,
                     sc, p, pairs, count, cap, eps, skip, bits, words);
}

// Candidate pairs of one or many scenes, culled and traced in one launch.  A
// wave takes one patch i and up to `chunk` columns j of its row (one group of
// patches against another, or all patches against all): 64 columns at a time
// pass the facing cull, the survivors' end points queue up in LDS, and 64 of
// them are traced together once they are there.  Bound by the walk: vector
// issue and the vector cache are each some 70 % busy.  The 8x8-room level's
// 2.57 G segments take 166 ms, 250 as rounds of list, trace and two atomics
// per visible pair.
//  - Segments of one wave share an end point and run to neighbouring patches.
//  - No pair list: it took 41 GB of traffic, 512 MB, and a hundred launches,
//    each with a tail.
//  - A wave sets its bits in row i alone, one atomic per word of 32 columns and
//    64 segments (two waves can meet in a word); k_bits_mirror then makes the
//    matrix symmetric.  An atomic per visible pair and direction was 3.2 G
//    atomics, half of them one per cache line.
template <int S>
__device__ __forceinline__ void pair_rows(const PairJob &J, int64_t gb, float eps, int32_t skip,
                                          uint32_t *s_stk, float4 *s_q, uint32_t *s_w) {
  int lo = 0, hi = J.n_tab - 1;
  while (lo < hi) {  // the entry whose blocks hold gb
    const int mid = (lo + hi + 1) >> 1;
    if (J.blk_pre[mid] <= gb) lo = mid;
    else hi = mid - 1;
  }
  const PvsEntry e = J.tab[lo];
  const int64_t local = gb - J.blk_pre[lo];
  const int ia = (int)(local / e.cpr);
  int col = (int)(local - (int64_t)ia * e.cpr) * J.chunk + (e.diag ? ia + 1 : 0);
  const int end = min(e.b_n, col + J.chunk);
  if (col >= end) return;
  const DevPatches &p = J.p;
  const int lane = (int)threadIdx.x;
  const int32_t *const mem = J.mem ? J.mem + e.b_off : nullptr;
  const int i = J.mem ? J.mem[e.a_off + ia] : ia;
  const float ix = p.ox[i], iy = p.oy[i], iz = p.oz[i];
  const float inx = p.nx[i], iny = p.ny[i], inz = p.nz[i];
  const float px = ix + eps * inx, py = iy + eps * iny, pz = iz + eps * inz;
  // the next 64 columns, loaded ahead of their use
  int j = -1;
  float jx = 0, jy = 0, jz = 0, jnx = 0, jny = 0, jnz = 0;
  auto fetch = [&](int at) {
    const int c = at + lane;
    j = c < end ? (mem ? mem[c] : c) : -1;
    if (j >= 0) {
      jx = p.ox[j], jy = p.oy[j], jz = p.oz[j];
      jnx = p.nx[j], jny = p.ny[j], jnz = p.nz[j];
    }
  };
  fetch(col);
  const uint64_t below = (1ull << lane) - 1ull;
  uint32_t head = 0, qn = 0, total = 0;  // survivors queued at [head, head + qn) mod 128
  BvhSpill<S, uint32_t> spill;
  BvhTracer<S, uint32_t> tr(J.sc, s_stk, lane, spill);
  uint32_t *const row = J.bits + (int64_t)i * J.words;
  uint8_t *const flag = J.flags + (int64_t)(i / kBitTile) * flag_stride(J.words);
  for (;;) {
    while (qn < 64u && col < end) {
      // the segment runs from the smaller patch index to the larger
      const bool ij = i < j;
      const float rx = ij ? ix : jx, ry = ij ? iy : jy, rz = ij ? iz : jz;
      const float qx = ij ? inx : jnx, qy = ij ? iny : jny, qz = ij ? inz : jnz;
      const float sx = ij ? jx : ix, sy = ij ? jy : iy, sz = ij ? jz : iz;
      const float tx = ij ? jnx : inx, ty = ij ? jny : iny, tz = ij ? jnz : inz;
      const float dx = sx - rx, dy = sy - ry, dz = sz - rz;
      const float di = (qx * dx + qy * dy) + qz * dz;
      const float dj = -((tx * dx + ty * dy) + tz * dz);
      const bool keep = j >= 0 && di > 0.0f && dj > 0.0f;
      const uint64_t m = __ballot(keep);
      if (keep)
        s_q[(head + qn + (uint32_t)__popcll(m & below)) & 127u] =
            make_float4(jx + eps * jnx, jy + eps * jny, jz + eps * jnz, __int_as_float(j));
      qn += (uint32_t)__popcll(m);
      col += 64;
      fetch(col);
    }
    const uint32_t n = min(qn, 64u);
    if (n == 0) break;
    __syncthreads();  // one wave: the queue is written before it is read
    const bool ray = (uint32_t)lane < n;
    const float4 q = s_q[(head + (uint32_t)lane) & 127u];
    const int jj = __float_as_int(q.w);
    const bool ij = i < jj;
    const bool vis =
        ray && segment_visible(J.sc, tr, ij ? px : q.x, ij ? py : q.y, ij ? pz : q.z,
                               ij ? q.x : px, ij ? q.y : py, ij ? q.z : pz, skip);
    head = (head + n) & 127u;
    qn -= n;
    total += n;
    // columns ascend, so a word's lanes are neighbours: they meet in the LDS
    // word of their run, which the run's first lane adds to the matrix
    const int w = jj >> 5;
    const int wl = __shfl_up(w, 1);
    const uint64_t heads = __ballot(ray && (lane == 0 || w != wl));
    const int run = __popcll(heads & (below | (1ull << lane))) - 1;
    s_w[lane] = 0u;
    __syncthreads();
    if (vis) atomicOr(&s_w[run], 1u << (jj & 31));
    __syncthreads();
    if ((heads >> lane) & 1ull) {
      const uint32_t v = s_w[run];
      if (v) {
        atomicOr(row + w, v);
        flag[w / kTileW] = 1;
      }
    }
  }
  // 64 counters, 64 bytes apart
  if (lane == 0 && total)
    atomicAdd(J.segs + 8 * (blockIdx.x & 63u), (unsigned long long)total);
}

// 6 waves per SIMD: before waves of several octants took scalar node loads,
// 186 ms on the level, against 189 with 5 and 198 with 8 (and spills)
template <int S>
__global__ __launch_bounds__(64, 6) void k_pair_rows(PairJob job, int64_t blk0, float eps,
                                                  int32_t skip, uint32_t xg) {
  __shared__ uint32_t s_stk[S * 64];
  __shared__ float4 s_q[128];
  __shared__ uint32_t s_w[64];
  pair_rows<S>(job, blk0 + xcd_group_chunk(blockIdx.x, gridDim.x, xg), eps, skip, s_stk, s_q,
               s_w);
}

// Block b (after the XCD remap) belongs to the job whose block range holds it
// (binary search over the jobs' first blocks; the index is the same for the
// whole wave, so the descriptor comes through scalar loads).
template <int S>
__global__ __launch_bounds__(64, 6) void k_pair_rows_jobs(const PairJob *__restrict__ jobs,
                                                       int n_jobs, int64_t blk0, float eps,
                                                       int32_t skip) {
  __shared__ uint32_t s_stk[S * 64];
  __shared__ float4 s_q[128];
  __shared__ uint32_t s_w[64];
  const int64_t b = blk0 + xcd_group_chunk(blockIdx.x, gridDim.x, kXcdGroup);
  int lo = 0, hi = n_jobs - 1;
  while (lo < hi) {  // last job with blk_begin <= b
    const int mid = (lo + hi + 1) >> 1;
    if (jobs[mid].blk_begin <= b) lo = mid;
    else hi = mid - 1;
  }
  const PairJob &J = jobs[__builtin_amdgcn_readfirstlane(lo)];
  pair_rows<S>(J, b - J.blk_begin, eps, skip, s_stk, s_q, s_w);
}

// Columns per wave.  Long rows waste less of their last 64 segments, short
// ones fill the chip: 16 K waves or more, of 256 to 8192 columns.
int pair_chunk(int64_t pairs) {
  const int64_t c = (pairs / 16384 + 63) / 64 * 64;
  return (int)std::min<int64_t>(8192, std::max<int64_t>(256, c));
}

// the traversal-stack entries kept in LDS follow the autotuned knob
#define VR_BY_LDS(X)                                                                       \
  switch (lds_entries) {                                                                   \
    case 2: X(2); break;                                                                   \
    case 4: X(4); break;                                                                   \
    case 6: X(6); break;                                                                   \
    case 10: X(10); break;                                                                 \
    case 12: X(12); break;                                                                 \
    case 16: X(16); break;                                                                 \
    case 24: X(24); break;                                                                 \
    default: X(8); break;                                                                  \
  }

void launch_pair_rows(const PairJob &job, int64_t n_blk, int64_t per, float eps, int32_t skip,
                      int lds_entries, int xcd_group, hipStream_t st) {
  for (int64_t b = 0; b < n_blk; b += per) {
    const dim3 grid((unsigned)std::min(per, n_blk - b));
#define VR_ROWS(S)                                                                        \
  hipLaunchKernelGGL((k_pair_rows<S>), grid, dim3(64), 0, st, job, b, eps, skip, (uint32_t)xcd_group)
    VR_BY_LDS(VR_ROWS)
#undef VR_ROWS
  }
}

void launch_pair_rows_jobs(const PairJob *jobs, int n_jobs, int64_t n_blk, int64_t per, float eps,
                           int32_t skip, int lds_entries, hipStream_t st) {
  for (int64_t b = 0; n_jobs > 0 && b < n_blk; b += per) {
    const dim3 grid((unsigned)std::min(per, n_blk - b));
#define VR_ROWS(S) \
  hipLaunchKernelGGL((k_pair_rows_jobs<S>), grid, dim3(64), 0, st, jobs, n_jobs, b, eps, skip)
    VR_BY_LDS(VR_ROWS)
#undef VR_ROWS
  }
}

// bits |= transpose(bits), in place.  A workgroup takes a tile of 512 x 512
// bits and its mirror image (64-byte row pieces, so whole memory accesses) if
// either holds a bit (flags): both go to LDS (rows 17 words apart: a column of
// words lies in 32 banks), half-waves exchange 32 x 32 bit blocks, transposed
// in 5 steps of the half a lane pairs up with, and the tiles go back.  Bound
// by the memory it moves: with a PVS most of the matrix is empty (on the
// 8x8-room level 9 rooms of 64 see a room): 9.0 ms without the flags, 1.8 with
// them, the counting pass 3.8 and 0.5.
constexpr int kMirrorS = kTileW + 1;

__device__ __forceinline__ uint32_t transpose32(uint32_t x, int l) {
  // rows and columns whose numbers differ in bit s change places, for each s
  uint32_t m = 0x0000ffffu;
#pragma unroll
  for (int s = 16; s >= 1; s >>= 1, m ^= m << s) {
    const uint32_t y = __shfl_xor(x, s);
    x = (l & s) ? (x & ~m) | ((y >> s) & m) : (x & m) | ((y & m) << s);
  }
  return x;
}

__global__ __launch_bounds__(256) void k_bits_mirror(uint32_t *__restrict__ bits,
                                                     uint8_t *__restrict__ flags, int64_t np,
                                                     int64_t words, uint32_t nt) {
  __shared__ uint32_t s_a[kBitTile * kMirrorS], s_b[kBitTile * kMirrorS];
  // tile (r, c), r <= c, of the upper triangle's row-by-row enumeration
  // folded in two: row r of the fold holds tiles (r, r..) and (nt-1-r, ..)
  const uint32_t w = nt + 1, f = blockIdx.x / w, x = blockIdx.x % w;
  uint32_t r = f, c = f + x;
  if (c >= nt) {
    r = nt - 1 - f;
    c = r + (x - (nt - f));
    if (r == f) return;  // the middle row of an odd count stands alone
  }
  const int64_t ra = (int64_t)r * kBitTile, rb = (int64_t)c * kBitTile;
  const int64_t wa = (int64_t)c * kTileW, wb = (int64_t)r * kTileW;
  const int t = (int)threadIdx.x, col = t & (kTileW - 1);
  const bool diag = r == c;
  uint8_t *const fa = flags + r * flag_stride(words) + c, *const fb = flags + c * flag_stride(words) + r;
  if ((*fa | *fb) == 0) return;  // read by all threads before the first barrier
#pragma unroll 8
  for (int k = t / kTileW; k < kBitTile; k += 256 / kTileW) {
    const uint32_t a = ra + k < np && wa + col < words ? bits[(ra + k) * words + wa + col] : 0u;
    const uint32_t b =
        !diag && rb + k < np && wb + col < words ? bits[(rb + k) * words + wb + col] : 0u;
    s_a[k * kMirrorS + col] = a;
    s_b[k * kMirrorS + col] = b;
  }
  __syncthreads();
  if (t == 0) *fa = *fb = 1;
  uint32_t *const s_m = diag ? s_a : s_b;
  const int half = t >> 5, l = t & 31;
  for (int q = half; q < kTileW * kTileW; q += 8) {
    const int br = q / kTileW, bc = q % kTileW;
    // both halves of a wave run the shuffles; of a diagonal tile's block pair
    // only one writes
    uint32_t *const pa = s_a + (32 * br + l) * kMirrorS + bc;
    uint32_t *const pb = s_m + (32 * bc + l) * kMirrorS + br;
    const uint32_t a = *pa | transpose32(*pb, l);
    const uint32_t b = transpose32(a, l);
    if (!diag || br <= bc) {
      *pb = b;
      *pa = a;
    }
  }
  __syncthreads();
#pragma unroll 8
  for (int k = t / kTileW; k < kBitTile; k += 256 / kTileW) {
    if (ra + k < np && wa + col < words) bits[(ra + k) * words + wa + col] = s_a[k * kMirrorS + col];
    if (!diag && rb + k < np && wb + col < words)
      bits[(rb + k) * words + wb + col] = s_b[k * kMirrorS + col];
  }
}

void launch_bits_mirror(uint32_t *bits, uint8_t *flags, int64_t np, int64_t words,
                        hipStream_t st) {
  if (np <= 0) return;
  const uint32_t nt = (uint32_t)((np + kBitTile - 1) / kBitTile);
  const uint32_t grid = (nt + 1) / 2 * (nt + 1);
  hipLaunchKernelGGL(k_bits_mirror, dim3(grid), dim3(256), 0, st, bits, flags, np, words,
                     nt);
}

// Chunks of 64 words (four tiles, one flag word) of a row that hold bits: the
// lanes look at 64 chunks' flags at once, f(chunk) runs for each with any
// set.
template <class F>
__device__ __forceinline__ void for_chunks(const uint8_t *flags, int64_t row, int64_t words,
                                           int lane, F f) {
  const uint32_t *fl = reinterpret_cast<const uint32_t *>(flags + row / kBitTile * flag_stride(words));
  const int64_t nq = (words + 63) / 64;
  for (int64_t q0 = 0; q0 < nq; q0 += 64) {
    uint64_t m = __ballot(q0 + lane < nq && fl[q0 + lane] != 0u);
    while (m) {
      const int64_t q = q0 + __ffsll((unsigned long long)m) - 1;
      m &= m - 1ull;
      f(q);
    }
  }
}

// one wave per row
__global__ __launch_bounds__(256) void k_row_count(const uint32_t *__restrict__ bits,
                                                   const uint8_t *__restrict__ flags, int64_t np,
                                                   int64_t words, int32_t *__restrict__ cnt) {
  const int lane = threadIdx.x & 63;
  const int64_t row =
      (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (row >= np) return;
  const uint32_t *rb = bits + row * words;
  int c = 0;
  for_chunks(flags, row, words, lane, [&](int64_t q) {
    const int64_t w = 64 * q + lane;
    if (w < words) c += __popc(rb[w]);
  });
  for (int off = 32; off >= 1; off >>= 1) c += __shfl_xor(c, off);
  if (lane == 0) cnt[row] = c;
}

void launch_row_count(const uint32_t *bits, const uint8_t *flags, int64_t np, int64_t words,
                      int32_t *cnt, hipStream_t st) {
  if (np <= 0) return;
  hipLaunchKernelGGL(k_row_count, dim3((unsigned)((np + 3) / 4)), dim3(256), 0, st, bits, flags,
                     np, words, cnt);
}

// Rows longest first, ties by index: a radix sort of the row numbers on their
// lengths, a byte a pass.  Waves of 1024 rows count their digits, one block
// scans the counts (digit by digit, waves in order), and the waves move their
// rows, 64 at a time in order: a row's rank among its wave's equal digits comes
// from ballots, so equal digits keep their order.  341,299 rows of up to 14k
// entries: 2 passes, under 0.2 ms; the host's sort took 16 ms with the GPU
// waiting.
constexpr int kSortRows = 1024;

__device__ __forceinline__ int sort_digit(int32_t len, int shift) {
  return 255 - ((len >> shift) & 255);  // descending
}

__global__ __launch_bounds__(64) void k_sort_count(const int32_t *__restrict__ cnt,
                                                   const int32_t *__restrict__ in, int64_t n,
                                                   int shift, int64_t nb,
                                                   int32_t *__restrict__ hist) {
  __shared__ int32_t h[256];
  const int lane = (int)threadIdx.x;
  for (int d = lane; d < 256; d += 64) h[d] = 0;
  __syncthreads();
  for (int r = 0; r < kSortRows; r += 64) {
    const int64_t i = (int64_t)blockIdx.x * kSortRows + r + lane;
    if (i < n) atomicAdd(&h[sort_digit(cnt[in ? in[i] : i], shift)], 1);
  }
  __syncthreads();
  for (int d = lane; d < 256; d += 64) hist[d * nb + blockIdx.x] = h[d];
}

// exclusive scan of m counts in place, one block
__global__ __launch_bounds__(1024) void k_sort_scan(int32_t *__restrict__ v, int64_t m) {
  __shared__ int32_t part[1024];
  const int t = (int)threadIdx.x;
  const int64_t per = (m + 1023) / 1024, b = min(m, t * per), e = min(m, b + per);
  int32_t s = 0;
  for (int64_t k = b; k < e; ++k) s += v[k];
  part[t] = s;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {
    const int32_t x = t >= d ? part[t - d] : 0;
    __syncthreads();
    part[t] += x;
    __syncthreads();
  }
  int32_t run = part[t] - s;
  for (int64_t k = b; k < e; ++k) {
    const int32_t x = v[k];
    v[k] = run;
    run += x;
  }
}

__global__ __launch_bounds__(64) void k_sort_move(const int32_t *__restrict__ cnt,
                                                  const int32_t *__restrict__ in, int64_t n,
                                                  int shift, int64_t nb,
                                                  const int32_t *__restrict__ at,
                                                  int32_t *__restrict__ out) {
  __shared__ int32_t s_at[256];
  const int lane = (int)threadIdx.x;
  for (int d = lane; d < 256; d += 64) s_at[d] = at[d * nb + blockIdx.x];
  __syncthreads();
  for (int r = 0; r < kSortRows; r += 64) {
    const int64_t i = (int64_t)blockIdx.x * kSortRows + r + lane;
    const bool live = i < n;
    const int32_t row = live ? (in ? in[i] : (int32_t)i) : 0;
    const int d = live ? sort_digit(cnt[row], shift) : 0;
    uint64_t same = __ballot(live);  // the lanes of this lane's digit
    for (int b = 0; b < 8; ++b) {
      const uint64_t m = __ballot((d >> b) & 1);
      same &= ((d >> b) & 1) ? m : ~m;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    const int32_t base = s_at[d];
    __syncthreads();  // one wave: all have read the digit's place
    if (live) {
      out[base + rank] = row;
      if (rank == 0) s_at[d] = base + __popcll(same);
    }
    __syncthreads();
  }
}

int64_t row_order_scratch(int64_t n) {
  return n + 256 * ((n + kSortRows - 1) / kSortRows);
}

void launch_row_order(const int32_t *cnt, int64_t n, int32_t longest, int32_t *order,
                      int32_t *scratch, hipStream_t st) {
  if (n <= 0) return;
  const int64_t nb = (n + kSortRows - 1) / kSortRows;
  int passes = 1;
  while (passes < 4 && (longest >> (8 * passes)) != 0) ++passes;
  int32_t *const buf[2] = {order, scratch}, *const hist = scratch + n;
  const int32_t *in = nullptr;
  for (int p = 0; p < passes; ++p) {
    int32_t *const out = buf[(passes - 1 - p) & 1];
    hipLaunchKernelGGL(k_sort_count, dim3((unsigned)nb), dim3(64), 0, st, cnt, in, n, 8 * p, nb,
                       hist);
    hipLaunchKernelGGL(k_sort_scan, dim3(1), dim3(1024), 0, st, hist, 256 * nb);
    hipLaunchKernelGGL(k_sort_move, dim3((unsigned)nb), dim3(64), 0, st, cnt, in, n, 8 * p, nb,
                       hist, out);
    in = out;
  }
}

__device__ __forceinline__ float form_factor(const DevPatches &p, int64_t i, int64_t j) {
  const float dx = p.ox[j] - p.ox[i], dy = p.oy[j] - p.oy[i], dz = p.oz[j] - p.oz[i];
  const float di = (p.nx[i] * dx + p.ny[i] * dy) + p.nz[i] * dz;
  const float dj = -((p.nx[j] * dx + p.ny[j] * dy) + p.nz[j] * dz);
  const float r2 = (dx * dx + dy * dy) + dz * dz;
  return ((di * dj) * p.area[j]) / ((VR_PI_F * r2) * r2);
}

// One wave per row, over the bit matrix row in chunks of 64 words (2048
// columns) that hold bits: each lane takes a word (the next chunk's is loaded
// ahead), the set bits' columns go to LDS at their rank in the chunk
// (ascending), and consecutive lanes then write consecutive entries (col and
// F_ij) to the CSR, so the stores are contiguous.  A wave per row that looked
// at every chunk in turn took 14.4 ms on the 8x8-room level, most of it the
// wait for 167 loads one after another; 7.0 now, against 3 for the stores.
__global__ __launch_bounds__(64) void k_row_fill(const uint32_t *__restrict__ bits,
                                                 const uint8_t *__restrict__ flags, int64_t np,
                                                 int64_t words, DevPatches p,
                                                 const int64_t *__restrict__ rp,
                                                 const int32_t *__restrict__ cnt,
                                                 int32_t *__restrict__ col,
                                                 float *__restrict__ coef) {
  __shared__ int32_t s_col[64 * 32];
  const int lane = (int)threadIdx.x;
  const int64_t row = blockIdx.x;
  if (row >= np) return;
  const uint32_t *rb = bits + row * words;
  const int64_t s = rp[row];
  int64_t run = 0;
  auto chunk = [&](int64_t q, uint32_t m) {
    const int64_t w = 64 * q + lane;
    const int pc = __popc(m);
    // inclusive wave scan of pc
    int inc = pc;
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(inc, off);
      if (lane >= off) inc += v;
    }
    const int tot = __shfl(inc, 63);
    if (tot == 0) return;
    int at = inc - pc;
    while (m) {
      const int bit = __ffs(m) - 1;
      m &= m - 1u;
      s_col[at++] = (int32_t)(w * 32 + bit);
    }
    __syncthreads();  // one wave: the chunk's columns are in LDS before they are read
    for (int k = lane; k < tot; k += 64) {
      const int32_t j = s_col[k];
      col[s + run + k] = j;
      coef[s + run + k] = form_factor(p, row, j);
    }
    __syncthreads();  // and read before the next chunk overwrites them
    run += tot;
  };
  int64_t held = -1;  // the chunk whose words are on their way
  uint32_t mh = 0;
  for_chunks(flags, row, words, lane, [&](int64_t q) {
    const int64_t w = 64 * q + lane;
    const uint32_t m = w < words ? rb[w] : 0u;
    if (held >= 0) chunk(held, mh);
    held = q;
    mh = m;
  });
  if (held >= 0) chunk(held, mh);
  const int64_t c = cnt[row], e = rp[row + 1];
  for (int64_t k = s + c + lane; k < e; k += 64) {
    col[k] = (int32_t)row;
    coef[k] = 0.0f;
  }
}

void launch_row_fill(const uint32_t *bits, const uint8_t *flags, int64_t np, int64_t words,
                     const DevPatches &p, const int64_t *rp, const int32_t *cnt, int32_t *col,
                     float *coef, hipStream_t st) {
  if (np <= 0) return;
  hipLaunchKernelGGL(k_row_fill, dim3((unsigned)np), dim3(64), 0, st, bits, flags, np, words, p, rp,
                     cnt, col, coef);
}

// FP64 row sum in wave order (lane owns p with (p/4)%64 == lane), butterfly
__global__ __launch_bounds__(256) void k_row_norm(int64_t n, const int64_t *__restrict__ rp,
                                                  float *__restrict__ coef,
                                                  double *__restrict__ row_sum, int normalize) {
  const int lane = threadIdx.x & 63;
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6;
  if (row >= n) return;
  const int64_t s = rp[row], e = rp[row + 1];
  double a = 0.0;
  for (int64_t k = s + 4 * lane; k < e; k += 256) {
    const float4 w = *reinterpret_cast<const float4 *>(coef + k);
    a = a + (double)w.x;
    a = a + (double)w.y;
    a = a + (double)w.z;
    a = a + (double)w.w;
  }
  for (int off = 32; off >= 1; off >>= 1) a = a + __shfl_xor(a, off);
  if (lane == 0) row_sum[row] = a;
  if (normalize && a > 1.0)
    for (int64_t k = s + lane; k < e; k += 64) coef[k] = (float)((double)coef[k] / a);
}

void launch_row_normalize(int64_t n, const int64_t *rp, float *coef, double *row_sum,
                          int normalize, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_row_norm, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, st, n, rp, coef,
                     row_sum, normalize);
}

}  // namespace vr
