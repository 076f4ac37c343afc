// GatherSampleLight: direct light at sample points from point, spot, surface,
// sun and sky-ambient lights, each term gated by TestLine visibility.  The
// per-light formulas and their operation order are those of the CPU
// restatement; lights are summed in list order.
#include "kernels.h"

namespace vr {

#define VR_MAX_TRACE_LENGTH_F ((float)(1.732050807569 * 32768.0))

// A spotlight cone's falloff, not inlined: FP64 pow takes twice the registers
// the walks need, which halved the waves in flight of every light's kernel.
__device__ __attribute__((noinline)) float cone_power(float dot2, float exponent) {
  return (float)pow((double)dot2, (double)exponent);
}

// One light other than sky ambient at a sample (p, n), whose visibility starts
// at s: false when it adds nothing, else the scale of its intensity and the
// segment's end.
__device__ __forceinline__ bool light_term(const vr_light &L, float px, float py, float pz,
                                           float nx, float ny, float nz, float sx, float sy,
                                           float sz, float &scale, float &ex, float &ey,
                                           float &ez) {
  if (L.type == VR_EMIT_SKYLIGHT) {
    const float MTL = VR_MAX_TRACE_LENGTH_F;
    const float dot = -((nx * L.normal[0] + ny * L.normal[1]) + nz * L.normal[2]);
    if (!(dot > 0.0f)) return false;
    ex = sx - MTL * L.normal[0];
    ey = sy - MTL * L.normal[1];
    ez = sz - MTL * L.normal[2];
    scale = dot;
    return true;
  }
  if (L.type != VR_EMIT_SURFACE && L.type != VR_EMIT_POINT && L.type != VR_EMIT_SPOTLIGHT)
    return false;
  ex = L.origin[0];
  ey = L.origin[1];
  ez = L.origin[2];
  const float lx = ex - px, ly = ey - py, lz = ez - pz;
  const float dist2 = (lx * lx + ly * ly) + lz * lz;
  if (!(dist2 > 0.0f)) return false;
  const float dist = __builtin_sqrtf(dist2);
  const float inv = 1.0f / dist;
  const float ux = lx * inv, uy = ly * inv, uz = lz * inv;
  const float dot = (nx * ux + ny * uy) + nz * uz;
  if (!(dot > 0.0f)) return false;
  if (L.type == VR_EMIT_SURFACE) {
    const float dot2 = -((L.normal[0] * ux + L.normal[1] * uy) + L.normal[2] * uz);
    if (!(dot2 > 0.0f)) return false;
    scale = (dot * dot2) / dist2;
    return true;
  }
  const float fd = dist < L.cap_distance ? dist : L.cap_distance;
  const float den = (L.constant_attn + L.linear_attn * fd) + L.quadratic_attn * (fd * fd);
  if (!(den > 0.0f)) return false;
  float fall = 1.0f / den;
  if (L.type == VR_EMIT_SPOTLIGHT) {
    const float dot2 = -((L.normal[0] * ux + L.normal[1] * uy) + L.normal[2] * uz);
    if (!(dot2 > L.stopdot2)) return false;
    if (dot2 <= L.stopdot) fall = fall * ((dot2 - L.stopdot2) / (L.stopdot - L.stopdot2));
    // the cone exponent in float64 then rounded: one rounding of a
    // near-exact power, so the value does not depend on a float powf
    if (L.exponent != 0.0f && L.exponent != 1.0f)
      fall = fall * cone_power(dot2, L.exponent);
  }
  if (L.end_fade > L.start_fade) {
    if (dist >= L.end_fade) return false;
    if (dist > L.start_fade) {
      const float x = (dist - L.start_fade) / (L.end_fade - L.start_fade);
      const float sm = (x * x) * (3.0f - 2.0f * x);
      fall = fall * (1.0f - sm);
    }
  }
  scale = dot * fall;
  return true;
}

constexpr int kSkyDirs = 162;
constexpr int kGatherBatch = 192;  // lights between two sums of a workgroup

// Direct light of 64 samples (one per lane) by the W waves of a workgroup: the
// waves take the lights, and the directions of a sky-ambient light, in turn
// and leave each one's visible lanes as a word in s_vis; wave 0 then adds the
// terms in list order, as one wave does alone (W = 1, no words).  A wave's
// lanes share the light or direction, so they start close together and head
// the same way.
//
// Bound by the walks' latency: a wave alone walks light after light.  60,013
// samples (938 groups on 1,024 SIMDs) with 9 lights and sky ambient took 2.07
// ms with one wave per group; the rule for W is at gather_waves.
template <int W, class Tracer>
__device__ void gather_group(const DevScene &sc, Tracer &tr, int wave, bool live, float px,
                             float py, float pz, float nx, float ny, float nz,
                             const vr_light *__restrict__ lights, int32_t n_lights,
                             const float *__restrict__ dirs, float eps, int32_t skip,
                             uint64_t *s_vis, float &r, float &g, float &b) {
  const float sx = px + eps * nx, sy = py + eps * ny, sz = pz + eps * nz;
  const float MTL = VR_MAX_TRACE_LENGTH_F;
  const int lane = (int)(threadIdx.x & 63);
  r = g = b = 0.0f;
  auto add = [&](const vr_light &L, float scale) {
    r = r + L.intensity[0] * scale;
    g = g + L.intensity[1] * scale;
    b = b + L.intensity[2] * scale;
  };
  auto cosine = [&](int k) {
    return (nx * dirs[3 * k] + ny * dirs[3 * k + 1]) + nz * dirs[3 * k + 2];
  };
  for (int32_t li = 0; li < n_lights;) {
    const vr_light &L = lights[li];
    const bool amb = L.type == VR_EMIT_SKYAMBIENT;
    // the walks of this turn: a sky-ambient light's directions, or this light
    // (W > 1: and the others up to the next sky-ambient one)
    int m = amb ? kSkyDirs : 1;
    if constexpr (W > 1)
      while (!amb && m < kGatherBatch && li + m < n_lights &&
             lights[li + m].type != VR_EMIT_SKYAMBIENT)
        ++m;
    float a = 0.0f, w = 0.0f, scale = 0.0f;
    for (int q = wave; q < m; q += W) {
      float ex, ey, ez;
      bool seen;
      if (amb) {
        scale = cosine(q);
        seen = scale > 0.0f;
        ex = sx + MTL * dirs[3 * q];
        ey = sy + MTL * dirs[3 * q + 1];
        ez = sz + MTL * dirs[3 * q + 2];
        if (W == 1 && seen) w = w + scale;
      } else {
        seen = light_term(lights[li + q], px, py, pz, nx, ny, nz, sx, sy, sz, scale, ex, ey, ez);
      }
      seen = seen && live && segment_visible(sc, tr, sx, sy, sz, ex, ey, ez, skip);
      if constexpr (W > 1) {
        const uint64_t word = __ballot(seen);
        if (lane == 0) s_vis[q] = word;
      } else if (seen) {
        if (amb) a = a + scale;
        else add(L, scale);
      }
    }
    if constexpr (W > 1) {
      __syncthreads();
      if (wave == 0)
        for (int q = 0; q < m; ++q) {
          const bool seen = ((s_vis[q] >> lane) & 1ull) != 0;
          if (amb) {
            const float ck = cosine(q);
            if (!(ck > 0.0f)) continue;
            w = w + ck;
            if (seen) a = a + ck;
          } else if (seen) {
            float ex, ey, ez;
            (void)light_term(lights[li + q], px, py, pz, nx, ny, nz, sx, sy, sz, scale, ex, ey,
                             ez);
            add(lights[li + q], scale);
          }
        }
      __syncthreads();
    }
    if (amb && w > 0.0f) add(L, a / w);
    li += amb ? 1 : m;
  }
}

template <int S, int W>
__global__ __launch_bounds__(64 * W, W >= 16 ? 4 : 6) void k_gather_lds(
    DevScene sc, DevSamples s, int64_t n, const vr_light *__restrict__ lights, int32_t n_lights,
    const float *__restrict__ dirs, float eps, int32_t skip, float *__restrict__ rgb) {
  __shared__ uint32_t s_stk[W * S * 64];
  __shared__ uint64_t s_vis[W > 1 ? kGatherBatch : 1];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t i0 = (int64_t)xcd_group_chunk(blockIdx.x, gridDim.x, kXcdGroup) * 64 +
                     (threadIdx.x & 63);
  const bool live = i0 < n;
  if (W == 1 && !live) return;
  const int64_t i = live ? i0 : n - 1;
  BvhSpill<S, uint32_t> spill;
  BvhTracer<S, uint32_t> tr(sc, s_stk + wave * S * 64, (int)(threadIdx.x & 63), spill);
  float r, g, b;
  gather_group<W>(sc, tr, wave, live, s.px[i], s.py[i], s.pz[i], s.nx[i], s.ny[i], s.nz[i],
                  lights, n_lights, dirs, eps, skip, s_vis, r, g, b);
  if (wave != 0 || !live) return;
  rgb[3 * i + 0] = r;
  rgb[3 * i + 1] = g;
  rgb[3 * i + 2] = b;
}

template <int D>
__global__ __launch_bounds__(256) void k_gather_plain(DevScene sc, DevSamples s, int64_t n,
                                                      const vr_light *__restrict__ lights,
                                                      int32_t n_lights,
                                                      const float *__restrict__ dirs, float eps,
                                                      int32_t skip, float *__restrict__ rgb) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  ScratchStack<D> st;
  KdTracer<D> tr(sc, st);
  float r, g, b;
  gather_group<1>(sc, tr, 0, true, s.px[i], s.py[i], s.pz[i], s.nx[i], s.ny[i], s.nz[i], lights,
                  n_lights, dirs, eps, skip, nullptr, r, g, b);
  rgb[3 * i + 0] = r;
  rgb[3 * i + 1] = g;
  rgb[3 * i + 2] = b;
}

// Many scenes' samples in one launch: block b (after the XCD remap) belongs
// to the job whose block range holds it (binary search; the job index is
// uniform per wave), and lane l gathers that job's sample
// (b - first block) * 64 + l from the job's scene and lights.
template <int S, int W>
__global__ __launch_bounds__(64 * W, W >= 16 ? 4 : 6) void k_gather_jobs(
    const GatherJob *__restrict__ jobs, int n_jobs, const float *__restrict__ dirs, float eps,
    int32_t skip) {
  __shared__ uint32_t s_stk[W * S * 64];
  __shared__ uint64_t s_vis[W > 1 ? kGatherBatch : 1];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t bk = (int64_t)xcd_group_chunk(blockIdx.x, gridDim.x, kXcdGroup);
  int lo = 0, hi = n_jobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (jobs[mid].blk_begin <= bk) lo = mid;
    else hi = mid - 1;
  }
  const int jx = __builtin_amdgcn_readfirstlane(lo);
  const GatherJob &J = jobs[jx];
  const int64_t i0 = (bk - J.blk_begin) * 64 + (threadIdx.x & 63);
  const bool live = i0 < J.n;
  if (W == 1 && !live) return;
  const int64_t i = live ? i0 : J.n - 1;
  BvhSpill<S, uint32_t> spill;
  BvhTracer<S, uint32_t> tr(J.sc, s_stk + wave * S * 64, (int)(threadIdx.x & 63), spill);
  const DevSamples &s = J.s;
  float r, g, b;
  gather_group<W>(J.sc, tr, wave, live, s.px[i], s.py[i], s.pz[i], s.nx[i], s.ny[i], s.nz[i],
                  J.lights, J.n_lights, dirs, eps, skip, s_vis, r, g, b);
  if (wave != 0 || !live) return;
  J.rgb[3 * i + 0] = r;
  J.rgb[3 * i + 1] = g;
  J.rgb[3 * i + 2] = b;
}

int64_t light_walks(const vr_light *lights, int32_t n_lights) {
  int64_t w = 0;
  for (int32_t k = 0; k < n_lights; ++k) w += lights[k].type == VR_EMIT_SKYAMBIENT ? kSkyDirs : 1;
  return w;
}

// Waves per group of 64 samples: the most of 1, 2, 4, 8, 16 that the walks of
// a group (lights, and 162 per sky-ambient one) can use, up to some 16 waves
// per SIMD in all.
static int gather_waves(int64_t groups, int64_t walks) {
  int w = 1;
  while (w < 16 && 2 * w <= walks && groups * w < 8192) w *= 2;
  return w;
}
#define VR_GATHER_S(X, W)                                                              \
  switch (lds_entries) {                                                               \
    case 2: X(2, W); break;                                                            \
    case 4: X(4, W); break;                                                            \
    case 6: X(6, W); break;                                                            \
    case 10: X(10, W); break;                                                          \
    case 12: X(12, W); break;                                                          \
    case 16: X(16, W); break;                                                          \
    case 24: X(24, W); break;                                                          \
    default: X(8, W); break;                                                           \
  }
#define VR_GATHER_W(X, w)                                                              \
  switch (w) {                                                                         \
    case 16: VR_GATHER_S(X, 16) break;                                                 \
    case 8: VR_GATHER_S(X, 8) break;                                                   \
    case 4: VR_GATHER_S(X, 4) break;                                                   \
    case 2: VR_GATHER_S(X, 2) break;                                                   \
    default: VR_GATHER_S(X, 1) break;                                                  \
  }

void launch_gather_jobs(const GatherJob *jobs, int n_jobs, int64_t total_blocks, int64_t walks,
                        const float *sky_dirs, float eps, int32_t skip, int lds_entries,
                        hipStream_t st) {
  if (n_jobs <= 0 || total_blocks <= 0) return;
#define VR_G_JOBS(S, W)                                                                  \
  hipLaunchKernelGGL((k_gather_jobs<S, W>), dim3((unsigned)total_blocks), dim3(64 * W), 0, st, \
                     jobs, n_jobs, sky_dirs, eps, skip)
  VR_GATHER_W(VR_G_JOBS, gather_waves(total_blocks, walks))
#undef VR_G_JOBS
}

// CanLeafTraceToSky (rad/lightmap/lightmap.go:425-451): one wave per leaf.
// The leaf's centre is float32(mins + maxs) * 0.5 per axis; lane l traces
// the segments from it to (a * -MAX_TRACE_LENGTH) + centre for the
// directions a = dirs[l], dirs[l + 64], dirs[l + 128] (< 162) with skip id
// -1, and the wave stops after the first round in which some lane's
// segment is visible (a miss, or a sky hit before any other).  "Any" does
// not depend on the order the directions are taken in.
template <class Tracer>
__device__ __forceinline__ void leaf_sky(const DevScene &sc, Tracer &tr, int64_t leaf,
                                         const int16_t *__restrict__ mins,
                                         const int16_t *__restrict__ maxs,
                                         const float *__restrict__ dirs,
                                         uint8_t *__restrict__ out) {
  const float cx = (float)((int32_t)mins[3 * leaf + 0] + (int32_t)maxs[3 * leaf + 0]) * 0.5f;
  const float cy = (float)((int32_t)mins[3 * leaf + 1] + (int32_t)maxs[3 * leaf + 1]) * 0.5f;
  const float cz = (float)((int32_t)mins[3 * leaf + 2] + (int32_t)maxs[3 * leaf + 2]) * 0.5f;
  const float nm = -VR_MAX_TRACE_LENGTH_F;
  uint8_t any = 0;
  for (int k0 = 0; k0 < 162; k0 += 64) {
    const int k = k0 + (int)threadIdx.x;
    bool vis = false;
    if (k < 162) {
      vis = segment_visible(sc, tr, cx, cy, cz, dirs[3 * k] * nm + cx,
                               dirs[3 * k + 1] * nm + cy, dirs[3 * k + 2] * nm + cz, -1);
    }
    if (__any(vis)) {
      any = 1;
      break;
    }
  }
  if (threadIdx.x == 0) out[leaf] = any;
}
template <int S>
__global__ __launch_bounds__(64) void k_leaf_sky(DevScene sc, const int16_t *__restrict__ mins,
                                                 const int16_t *__restrict__ maxs, int64_t n,
                                                 const float *__restrict__ dirs,
                                                 uint8_t *__restrict__ out) {
  __shared__ uint32_t s_stk[S * 64];
  const int64_t leaf = (int64_t)xcd_group_chunk(blockIdx.x, gridDim.x, kXcdGroup);
  if (leaf >= n) return;
  BvhSpill<S, uint32_t> spill;
  BvhTracer<S, uint32_t> tr(sc, s_stk, (int)threadIdx.x, spill);
  leaf_sky(sc, tr, leaf, mins, maxs, dirs, out);
}
// scenes too large for the hierarchy's 32-bit offsets
template <int D>
__global__ __launch_bounds__(64) void k_leaf_sky_kd(DevScene sc, const int16_t *__restrict__ mins,
                                                    const int16_t *__restrict__ maxs, int64_t n,
                                                    const float *__restrict__ dirs,
                                                    uint8_t *__restrict__ out) {
  if ((int64_t)blockIdx.x >= n) return;
  ScratchStack<D> st;
  KdTracer<D> tr(sc, st);
  leaf_sky(sc, tr, blockIdx.x, mins, maxs, dirs, out);
}

void launch_leaf_sky(const DevScene &sc, const int16_t *mins, const int16_t *maxs, int64_t n,
                     const float *sky_dirs, uint8_t *out, hipStream_t st) {
  if (n <= 0) return;
  if (!sc.has_bvh) {
    hipLaunchKernelGGL((k_leaf_sky_kd<kStackDepth>), dim3((unsigned)n), dim3(64), 0, st, sc, mins,
                       maxs, n, sky_dirs, out);
    return;
  }
#define VR_LEAFSKY(S)                                                                      \
  hipLaunchKernelGGL((k_leaf_sky<S>), dim3((unsigned)n), dim3(64), 0, st, sc, \
                     mins, maxs, n, sky_dirs, out)
  switch (tuning().trace_lds_entries) {
    case 2: VR_LEAFSKY(2); break;
    case 4: VR_LEAFSKY(4); break;
    case 6: VR_LEAFSKY(6); break;
    case 10: VR_LEAFSKY(10); break;
    case 12: VR_LEAFSKY(12); break;
    case 16: VR_LEAFSKY(16); break;
    case 24: VR_LEAFSKY(24); break;
    default: VR_LEAFSKY(8); break;
  }
#undef VR_LEAFSKY
}

void launch_gather_light(const DevScene &sc, const DevSamples &s, int64_t n,
                         const vr_light *lights, int32_t n_lights, int64_t walks,
                         const float *sky_dirs, float eps, int32_t skip, float *rgb, int path,
                         int lds_entries, hipStream_t st) {
  if (n <= 0) return;
  if (path == VR_PATH_PLAIN || !sc.has_bvh)
    hipLaunchKernelGGL(k_gather_plain<kStackDepth>, dim3((unsigned)((n + 255) / 256)), dim3(256),
                       0, st, sc, s, n, lights, n_lights, sky_dirs, eps, skip, rgb);
  else {
    // the traversal-stack entries kept in LDS: the caller's (autotuned) knob
#define VR_GATHER(S, W)                                                                       \
  hipLaunchKernelGGL((k_gather_lds<S, W>), dim3((unsigned)((n + 63) / 64)), dim3(64 * W), 0,  \
                     st, sc, s, n, lights, n_lights, sky_dirs, eps, skip, rgb)
    VR_GATHER_W(VR_GATHER, gather_waves((n + 63) / 64, walks))
#undef VR_GATHER
  }
}

}  // namespace vr
