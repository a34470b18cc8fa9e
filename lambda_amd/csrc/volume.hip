// Volumetric shade stage of the wavefront: one launch processes one iteration of
// VolumetricPathIntegrator::Li (VolumetricPathIntegrator.cpp:20-162) or
// MISVolumetricPathIntegrator::Li (MISVolumetricPathIntegrator.cpp:71-215) for every live path,
// after the extend stage has traced the path's ray.
//
// Per path and launch:
//   1. the light reached by the previous vertex's BSDF / phase sample (MIS), deferred to here
//      because that sample's ray is the continuation ray the extend stage just traced;
//      with kFlagTrMIS the lookup continues through pass-through surfaces multiplying Tr;
//   2. bounce-0 emission (camera rays, also after pass-through surfaces at depth 0);
//   3. inside a medium: distance sampling (VOLPATH) or the light-point / distance /
//      equiangular triple with both medium points' direct light (MIS_VOLPATH);
//   4. otherwise the surface vertex (NEE + BSDF sample) or a pass-through boundary;
//   5. Russian roulette, then the continuation is appended to the next queue.
// Traced inline, all rays of a vertex run under the divergent masks of the shading code (9 of 64
// lanes active in the fog room, measured), at the shading code's occupancy of two waves per SIMD.
// For the corrected estimator the rays therefore run in kernels of their own: step 1 in k_vol_light
// before, NEE visibility in k_vol_shadow after k_shade_vol, each with the block's rays gathered into
// full waves. The faithful estimator and the adjoint replay need a ray's result inside the vertex and
// trace inline, and so do the phase-sampled lookups of MIS_VOLPATH's medium points (kVolSplitLookup, scenes
// with emissive meshes or a sky). VALU instructions in the fog room, a pass: 2.6e9 in one kernel; 0.29e9
// here, 0.30e9 in k_vol_light and 0.48e9 in k_vol_shadow, at 28, 20 and 20 lanes. Fog room (301 x 211, 16
// spp) 13.8 -> 10.1 ms, media workload (1024 x 1024, 4 spp, 128^3 grid) 21.7 -> 17.3 ms.
#include "volume_kernel.h"

namespace lgpu {

namespace {

// Scene::IntersectTr (Scene.cpp:45-81) as media.h's, with the hit records of the crossed surfaces
// reduced to what the walk needs. t, u, v, bi: the last hit, o: the start of its segment.
struct TrWalk {
  V3 o;
  float t, u, v, tFar = INFINITY;  // tFar: distance walked when the walk ended on a surface
  uint32_t bi = kNone;
  Spec Tr;
  bool si = false, left = false;
};
__device__ inline void WalkTr(const DevScene &sc, TrWalk &w, V3 d, uint32_t med, float maxT, const VmCtx &vm,
                              const TraceCtx &tc, bool haveFirst) {
  float tFar = 0.f;
  for (int k = 0; k < 256; ++k) {
    uint32_t prim;
    if (!(k == 0 && haveFirst) &&
        !Trace4Closest(sc, w.o, d, 0.f, INFINITY, &w.t, &w.u, &w.v, &prim, &w.bi, tc.stk, tc.spill)) {
      w.left = true;
      return;
    }
    const float4 *tp = reinterpret_cast<const float4 *>(sc.tris + w.bi);
    const float4 w1 = tp[1], w2 = tp[2];
    const V3 n = Norm(Cross(v3(w1.x, w1.y, w1.z), v3(w2.x, w2.y, w2.z)));
    float seg = w.t;
    tFar += seg;
    const bool terminate = maxT >= 0.f && tFar > maxT;
    if (terminate) {
      const float delta = tFar - maxT;
      tFar -= delta;
      seg -= delta;
    }
    if (med != kNone) w.Tr = w.Tr * MediumTr(sc, sc.media[med], w.o, d, seg, vm);
    const MaterialRec mat = sc.materials[sc.meshes[__float_as_uint(w1.w)].material];
    w.tFar = seg;
    if (terminate || mat.lobe != kNone || mat.emission != kNone) {
      w.tFar = tFar;
      w.si = true;
      return;
    }
    med = GetMedium(mat, d, n);
    const V3 p = v3(w.o.x + d.x * w.t, w.o.y + d.y * w.t, w.o.z + d.z * w.t);
    w.o = p + n * (Dot(n, d) < 0 ? -kSurfaceEpsilon : kSurfaceEpsilon);
  }
}

__device__ inline void WaveLengths(VmCtx &vm, const DevScene &sc, uint32_t mode, float l0) {
  vm.mode = (int)mode;
  vm.texels = sc.texels; vm.textures = sc.textures; vm.consts = sc.consts; vm.code = sc.code;
  for (int k = 0; k < 4; ++k) {
    float l = l0 + 117.5f * (float)k;
    if (l >= 830.f) l -= 470.f;
    vm.lam[k] = mode ? l : 0.f;
  }
  vm.woLy = 0.f;
  vm.eta = 0.f;
  vm.medium = 0;
}

// The block's threads whose flag is set, in order: their indices go to list, the count is returned.
// Every thread of the block calls it; it begins and ends with a barrier. cnt: kBlock / 64 words.
__device__ inline uint32_t BlockGather(bool take, uint32_t *cnt, uint16_t *list, uint32_t first) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint64_t m = __ballot(take);
  __syncthreads();
  if (lane == 0) cnt[wv] = (uint32_t)__popcll(m);
  __syncthreads();
  uint32_t before = first, total = first;
  for (int w = 0; w < kBlock / 64; ++w) {
    if (w < wv) before += cnt[w];
    total += cnt[w];
  }
  if (take) list[before + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)threadIdx.x;
  __syncthreads();
  return total;
}

// Step 1 for the block's paths that reach a light or cross a boundary: the light reached by the
// previous vertex's sampled direction, added to the sample's radiance. Paths whose lookup has to walk
// on through pass-through surfaces come first, so the walking waves are full.
// Five waves per SIMD, here and in k_vol_shadow: media workload 15.9 ms at four, 15.4 at five and at six.
template <int kPrograms>
__global__ void __launch_bounds__(kBlock, 5)
    k_vol_light(const DevScene *__restrict__ scp, RenderParams rp, PathState ps, SampleState ss, uint32_t n,
                const uint32_t *np, uint32_t *spillBase, BounceSlot *slot) {
  if (slot) Stamp(&slot->shade);
  const DevScene &sc = *scp;
  __shared__ uint32_t stk[kLdsStack][kBlock];
  __shared__ uint32_t cnt[kBlock / 64];
  __shared__ uint16_t list[kBlock];
  if (np) n = *np;
  const uint32_t base = blockIdx.x * kBlock, own = base + threadIdx.x;
  if (base >= n) return;
  bool walk = false, look = false;
  if (own < n) {
    const uint32_t flags = ps.ids[own].w, hb = __float_as_uint(ps.hit[own].w);
    if (!(flags & (kFlagCamera | kFlagNoEmit))) {
      if (hb == kNone) {
        look = sc.has_env;
      } else {
        walk = (flags & kFlagTrMIS) && (sc.tris[hb].key & (kShadeKeys - 1)) == 1u;
        look = !walk && sc.meshes[__float_as_uint(reinterpret_cast<const float4 *>(sc.tris + hb)[1].w)].mesh_light != kNone;
      }
    }
  }
  const uint32_t walks = BlockGather(walk, cnt, list, 0u);
  const uint32_t total = BlockGather(look, cnt, list, walks);
  if (threadIdx.x >= total) return;
  const uint32_t i = base + list[threadIdx.x];
  const uint4 aux = ps.aux[i];
  const uint32_t flags = ps.ids[i].w;
  const float4 ro4 = ps.ray_o[i], rd4 = ps.ray_d[i], hr = ps.hit[i];
  const V3 rd = ToV3(rd4);
  VmCtx vm;
  WaveLengths(vm, sc, rp.mode, ro4.w);
  vm.eta = rd4.w;
  VmAtHit(vm, 0.f, 0.f, v3(0.f, 0.f, 0.f), v3(0.f, 0.f, 0.f));
  TrWalk w;
  w.o = ToV3(ro4);
  w.t = hr.x; w.u = hr.y; w.v = hr.z; w.bi = __float_as_uint(hr.w);
  w.Tr = S(1.f);
  w.si = w.bi != kNone;
  w.tFar = hr.x;
  if ((flags & kFlagTrMIS) && w.si) {
    w.si = false;
    WalkTr(sc, w, rd, aux.w, -1.f, vm, TraceCtx{stk, spillBase + (size_t)own * sc.spill_words}, true);
  }
  Hit h;
  if (w.si) {
    ProcessHit(sc, w.o, rd, w.t, w.u, w.v, w.bi, true, h);
    h.tFar = w.tFar;
  }
  const float4 mis = ps.mis[i], pn = ps.prev_n[i];
  vm.medium = pn.w != 0.f;  // looked up for a medium interaction
  const Spec C = MisLight<kPrograms>(sc, aux.y, mis.y, ToV3(ps.prev_p[i]), ToV3(pn), w.si, h, w.bi, rd, mis.x,
                                     (flags & kFlagSpecular) != 0, false, vm, true);
  const Spec c = S4(ps.beta[i]) * (C * w.Tr * mis.w);
  if (IsBlack(c, 1)) return;
  float4 L = ss.L[aux.x];
  L.x += c.c[0]; L.y += c.c[1]; L.z += c.c[2]; L.w += c.c[3];
  ss.L[aux.x] = L;
}

// The visibility rays of the block's vertices (VolRays), slot by slot: a slot's rays are gathered
// into full waves, and a path's second ray adds to its radiance after its first.
__global__ void __launch_bounds__(kBlock, 5)
    k_vol_shadow(const DevScene *__restrict__ scp, RenderParams rp, PathState ps, SampleState ss, uint32_t n,
                 const uint32_t *np, uint32_t *spillBase, int slots, BounceSlot *slot, BounceSlot *host) {
  if (slot && blockIdx.x == 0 && threadIdx.x == 0) Publish(slot, host);  // closes the bounce
  const DevScene &sc = *scp;
  __shared__ uint32_t stk[kLdsStack][kBlock];
  __shared__ uint32_t cnt[kBlock / 64];
  __shared__ uint16_t list[kBlock];
  if (np) n = *np;
  const uint32_t base = blockIdx.x * kBlock, own = base + threadIdx.x;
  if (base >= n) return;
  const uint32_t ownBits = own < n ? __float_as_uint(ps.hit[own].z) : 0u;
  const TraceCtx tc{stk, spillBase + (size_t)own * sc.spill_words};
  for (int s = 0; s < slots; ++s) {
    const uint32_t total = BlockGather((ownBits >> s) & 1u, cnt, list, 0u);
    if (threadIdx.x >= total) continue;
    const uint32_t i = base + list[threadIdx.x], sid = ps.aux[i].x;
    const float4 o4 = (s ? ps.mis : ps.ray_o)[i], d4 = (s ? ps.prev_p : ps.ray_d)[i], hr = ps.hit[i];
    const V3 d = ToV3(d4);
    TrWalk w;
    w.o = ToV3(o4);
    w.Tr = S(1.f);
    bool visible;
    if (sc.num_media > 0) {
      VmCtx vm;
      WaveLengths(vm, sc, rp.mode, ss.lambda0[sid]);
      WalkTr(sc, w, d, __float_as_uint(s ? hr.y : hr.x), o4.w, vm, tc, false);
      const bool escape = ((__float_as_uint(hr.z) >> s) & kRayEscape) != 0u;
      visible = escape ? !w.si : (w.left || w.tFar > d4.w);
    } else {
      float t, u, v;
      uint32_t prim, bi;
      visible = !Trace<true, false>(sc, w.o, d, 0.f, o4.w, &t, &u, &v, &prim, &bi, tc.stk, tc.spill, nullptr);
    }
    if (!visible) continue;
    const Spec c = S4((s ? ps.prev_n : ps.beta)[i]) * w.Tr;
    float4 L = ss.L[sid];
    L.x += c.c[0]; L.y += c.c[1]; L.z += c.c[2]; L.w += c.c[3];
    ss.L[sid] = L;
  }
}

// Closes a bounce whose shading is a single kernel.
__global__ void k_publish(BounceSlot *slot, BounceSlot *host) {
  slot->shadows = wall_clock64();
  Publish(slot, host);
}

}  // namespace

void LaunchVolFaithful(uint32_t blocks, hipStream_t stream, const DevScene &sc, const RenderParams &rp,
                       PathState ps, SampleState ss, uint32_t n, Queues q, uint32_t *spill, const uint32_t *np,
                       BounceSlot *slot);
void LaunchVolAdjoint(uint32_t blocks, hipStream_t stream, const DevScene *scp, int programs, const RenderParams &rp,
                      PathState ps, SampleState ss, uint32_t n, Queues q, uint32_t *spill, const AdjRefs &ar,
                      const uint32_t *np, BounceSlot *slot);

uint32_t LaunchShadeVol(uint32_t blocks, hipStream_t stream, const DevScene &sc, const DevScene *scp, const RenderParams &rp,
                        PathState ps, SampleState ss, uint32_t n, Queues q, uint32_t *spill, const AdjRefs *adj,
                        const uint32_t *np, BounceSlot *slot, BounceSlot *host) {
  const int programs = (int)sc.has_programs;
  if (adj || !rp.corrected) {
    if (adj) LaunchVolAdjoint(blocks, stream, scp, programs, rp, ps, ss, n, q, spill, *adj, np, slot);
    else LaunchVolFaithful(blocks, stream, sc, rp, ps, ss, n, q, spill, np, slot);
    if (slot) hipLaunchKernelGGL(k_publish, dim3(1), dim3(1), 0, stream, slot, host);
    return 1;
  }
  const dim3 g(blocks), b(kBlock);
  const bool lights = sc.has_mesh_lights || sc.has_env;  // lights that a sampled direction can reach
  const bool misVol = rp.integrator == LGPU_INTEGRATOR_MIS_VOLPATH;
  const AdjRefs none{};
  BounceSlot *first = lights ? nullptr : slot;  // the stage's start is stamped by its first kernel
#define LGPU_VOL_LIGHT(kLevel) \
  hipLaunchKernelGGL(k_vol_light<kLevel>, g, b, 0, stream, scp, rp, ps, ss, n, np, spill, slot)
#define LGPU_VOL_SHADE(kLevel, kMode) \
  hipLaunchKernelGGL((k_shade_vol<kLevel, kMode>), g, b, 0, stream, scp, rp, ps, ss, n, np, q, spill, none, first)
  if (lights) {
    if (programs == kVmPrograms) LGPU_VOL_LIGHT(kVmPrograms);
    else if (programs == kTexPrograms) LGPU_VOL_LIGHT(kTexPrograms);
    else LGPU_VOL_LIGHT(kNoPrograms);
  }
  if (misVol && lights) {
    if (programs) LGPU_VOL_SHADE(kVmPrograms, kVolSplitLookup);
    else LGPU_VOL_SHADE(kNoPrograms, kVolSplitLookup);
  } else if (programs == kVmPrograms) {
    LGPU_VOL_SHADE(kVmPrograms, kVolSplit);
  } else if (programs == kTexPrograms) {
    LGPU_VOL_SHADE(kTexPrograms, kVolSplit);
  } else {
    LGPU_VOL_SHADE(kNoPrograms, kVolSplit);
  }
#undef LGPU_VOL_LIGHT
#undef LGPU_VOL_SHADE
  hipLaunchKernelGGL(k_vol_shadow, g, b, 0, stream, scp, rp, ps, ss, n, np, spill, misVol ? 2 : 1, slot, host);
  return lights ? 3 : 2;
}

}  // namespace lgpu
