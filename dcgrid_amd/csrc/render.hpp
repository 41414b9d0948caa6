// render.hpp — gfx950 ray marcher over the simulation fields: FluidSimulation::render
// (src/fluid_simulation.h:19) for both grids, following src/raymarching.cuh:63-275 with the
// samplers of src/dcgrid/dcgrid_rendering.cu:6-64 and src/uniformgrid/uniformgrid_rendering.cu:5-47.
//
// One, 4 or 16 lanes per ray (MarchGroup, marchRoute). Every float operation is written out in the order of the
// reference's helper_math expressions, with correctly rounded division and square root and the
// library's own deterministic exp, so the image equals the oracle's restatement bit for bit.
// Deliberate differences: normalize divides by the length (helper_math multiplies by rsqrtf); the
// exp of the Beer-Lambert terms is expDet, 0 below -87; the apron coordinates of a precise sample
// are clamped into the block's apron (the reference indexes them unchecked; they only leave it
// for positions outside the domain); with terrain solids the scene distance is half the height
// above the terrain (the reference's scene is the sphere alone).
#pragma once

#include <float.h>

#include <utility>

#include "dcg_device.hpp"

namespace dcg {

// MarchAux (src/raymarching.cuh:18-41): the last sample's cell, trilinear fraction, the 8
// corner cells and the density there.
struct MarchAux {
  int3 ipos;
  float3 frac;
  uint32_t cell[8];
  float density;
};

template <class T>
__device__ __forceinline__ float marchInterp(const T* __restrict__ v, const MarchAux& a) {
  const float dx = a.frac.x, dxi = 1.f - dx;
  const float c00 = (float)v[a.cell[0]] * dxi + (float)v[a.cell[4]] * dx;
  const float c01 = (float)v[a.cell[1]] * dxi + (float)v[a.cell[5]] * dx;
  const float c10 = (float)v[a.cell[2]] * dxi + (float)v[a.cell[6]] * dx;
  const float c11 = (float)v[a.cell[3]] * dxi + (float)v[a.cell[7]] * dx;
  const float dy = a.frac.y, dyi = 1.f - dy;
  const float c0 = c00 * dyi + c10 * dy;
  const float c1 = c01 * dyi + c11 * dy;
  return c0 * (1.f - a.frac.z) + c1 * a.frac.z;
}
template <class V>
__device__ __forceinline__ float3 marchInterp3(const V* __restrict__ v, const MarchAux& a) {
  float3 c[8];
#pragma unroll
  for (int k = 0; k < 8; k++) c[k] = v[a.cell[k]];
  const float dx = a.frac.x, dxi = 1.f - dx, dy = a.frac.y, dyi = 1.f - dy, dz = a.frac.z, dzi = 1.f - dz;
  auto lerp3 = [](float3 p, float pw, float3 q, float qw) {
    return make_float3(p.x * pw + q.x * qw, p.y * pw + q.y * qw, p.z * pw + q.z * qw);
  };
  const float3 c00 = lerp3(c[0], dxi, c[4], dx), c01 = lerp3(c[1], dxi, c[5], dx);
  const float3 c10 = lerp3(c[2], dxi, c[6], dx), c11 = lerp3(c[3], dxi, c[7], dx);
  const float3 c0 = lerp3(c00, dyi, c10, dy), c1 = lerp3(c01, dyi, c11, dy);
  return lerp3(c0, dzi, c1, dz);
}

__device__ __forceinline__ float3 v3add(float3 a, float3 b) { return make_float3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ float3 v3sub(float3 a, float3 b) { return make_float3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ float3 v3mul(float3 a, float s) { return make_float3(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ float v3len(float3 a) { return __builtin_sqrtf(a.x * a.x + a.y * a.y + a.z * a.z); }
__device__ __forceinline__ float3 v3norm(float3 a) {
  const float l = v3len(a);
  return make_float3(a.x / l, a.y / l, a.z / l);
}
// exp of a Beer-Lambert exponent (__expf in the reference).
__device__ __forceinline__ float marchExp(float x) { return x < -87.f ? 0.f : expDet(x); }
// densityToAlpha (src/raymarching.cuh:43-46)
__device__ __forceinline__ float densityToAlpha(const dcg_params& P, float distance, float density) {
  return 1.f - marchExp(-distance * P.dx * density);
}
// mix (src/utils/colors.cuh:5-14): front-to-back compositing.
__device__ __forceinline__ void marchMix(float3 src, float srcA, float3& dst, float& dstA) {
  if (srcA > 1e-6f) {
    const float impact = (1.f - dstA) * srcA;
    const float den = dstA + impact;
    dst = make_float3((dst.x * dstA + src.x * impact) / den, (dst.y * dstA + src.y * impact) / den,
                      (dst.z * dstA + src.z * impact) / den);
    dstA = dstA + impact;
  }
}
// rayDomainIntersections (src/raymarching.cuh:48-78)
__device__ __forceinline__ bool rayDomain(const dcg_params& P, float& dNear, float& dFar, float3 o, float3 inv) {
  const float cx = (float)P.gx * .5f, cy = (float)P.gy * .5f, cz = (float)P.gz * .5f;
  const float nx = inv.x * (o.x - cx), ny = inv.y * (o.y - cy), nz = inv.z * (o.z - cz);
  const float kx = fabsf(inv.x) * cx, ky = fabsf(inv.y) * cy, kz = fabsf(inv.z) * cz;
  const float t1x = -nx - kx, t1y = -ny - ky, t1z = -nz - kz;
  const float t2x = -nx + kx, t2y = -ny + ky, t2z = -nz + kz;
  dNear = fmaxf(fmaxf(t1x, t1y), t1z);
  dFar = fminf(fminf(t2x, t2y), t2z);
  return dNear < dFar && dFar > 0.f;
}
// sceneSDF (src/sdf.cuh:8-22): the sphere of the additional solids, or half the height above
// the terrain (extension).
__device__ __forceinline__ float sceneSDF(const dcg_params& P, float3 p) {
  if (P.solid_mode == DCG_SOLID_TERRAIN) return .5f * (p.y - terrainHeight(P, p.x, p.z));
  const float cx = (float)P.gx * .5f, cy = (float)P.gy * .45f, cz = (float)P.gz * .5f;
  const float r = 2000.f * P.rdx;
  const float dx = p.x - cx, dy = p.y - cy, dz = p.z - cz;
  return __builtin_sqrtf(dx * dx + dy * dy + dz * dz) - r;
}
// estimateNormal (src/sdf.cuh:24-33)
__device__ __forceinline__ float3 sceneNormal(const dcg_params& P, float3 p) {
  const float e = 1e-4f;
  return v3norm(make_float3(sceneSDF(P, make_float3(p.x + e, p.y, p.z)) - sceneSDF(P, make_float3(p.x - e, p.y, p.z)),
                            sceneSDF(P, make_float3(p.x, p.y + e, p.z)) - sceneSDF(P, make_float3(p.x, p.y - e, p.z)),
                            sceneSDF(P, make_float3(p.x, p.y, p.z + e)) - sceneSDF(P, make_float3(p.x, p.y, p.z - e))));
}

// The march's lanes per ray. A ray is a long serial chain (up to two samples per cell of its path,
// each dense one with a shadow march of up to 100 samples), and an image has few rays for this chip:
// one thread per pixel gives a 256 x 256 image one wavefront per SIMD, bound by the latency of the
// dependent loads of its slowest ray (the time hardly depended on the resolution). GL = 16 lanes (one
// DPP row, or a quad of 4) take a ray together: each lane samples its own step of the next GL, and the sums that have to run
// in the ray's order (positions, optical depth, compositing) are formed by every lane alike from
// its neighbours' values, in the same order and with the same float operations as by one thread.
// GL = 1 is the plain loop, for images that fill the chip by themselves and the debug slices (marchRoute
// draws the line).
// Measured (MI355X, one thread per ray -> 16 lanes, 256 x 256): plume on the 256^3 grid 34 -> 3.0 ms,
// on the 512^3 grid 51 -> 3.7 ms, 4^3 blocks with a solid sphere 35 -> 3.2 ms, dense 64^3 grid
// 1.2 -> 0.30 ms, terrain 2.4 -> 0.72 ms.
template <int GL>
struct MarchGroup {
  static_assert(GL == 1 || GL == 4 || GL == 16, "one thread, one DPP quad or one DPP row per ray");
  static __device__ __forceinline__ int lane() { return GL == 1 ? 0 : (int)(threadIdx.x & (GL - 1)); }
  // Value of lane J of the group.
  template <int J>
  static __device__ __forceinline__ float from(float v) {
    if (GL == 1) return v;
    // quad_perm:[J,J,J,J] or row_newbcast:J; the lanes of a group run the march in lockstep, so
    // lane J is active
    constexpr int ctrl = GL == 4 ? 0x55 * J : 0x150 + J;
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xF, 0xF, true));
  }
  // Value of lane j, the same j in the whole group.
  static __device__ __forceinline__ float at(float v, int j) { return GL == 1 ? v : __shfl(v, j, GL); }
  // Bit k: lane k's condition.
  static __device__ __forceinline__ uint32_t ballot(bool c) {
    if (GL == 1) return c ? 1u : 0u;
    return (uint32_t)(__ballot(c) >> (threadIdx.x & (64u - GL))) & ((1u << GL) - 1u);
  }
  // op(J) for J = 0 .. GL - 1, J a constant.
  template <class Op, int... J>
  static __device__ __forceinline__ void eachOf(Op op, std::integer_sequence<int, J...>) {
    (op(std::integral_constant<int, J>{}), ...);
  }
  template <class Op>
  static __device__ __forceinline__ void each(Op op) {
    eachOf(op, std::make_integer_sequence<int, GL>{});
  }
};

// lightmarch (src/raymarching.cuh:80-121), the solid scene's part: 0 = fully shadowed.
__device__ __forceinline__ float sceneLight(const dcg_params& P, const dcg_render_params& R, float3 origin, float3 sun) {
  float lt = 1.f;
  if (R.solids && P.enable_additional_solids) {
    float dScene = 0.f;
    for (int i = 0; i < 100; i++) {
      const float sdf = sceneSDF(P, v3add(origin, v3mul(sun, dScene)));
      lt = fminf(lt, (sdf / dScene) / .06f);
      if (lt <= 1e-2f) return 0.f;
      dScene = dScene + sdf;
    }
  }
  return lt;
}
// lightmarch, the fluid's part, after the scene's `lt`: each lane of the group samples one step.
template <int GL, class S>
__device__ __forceinline__ float fluidLight(const S& smp, const dcg_params& P, const dcg_render_params& R, float3 origin,
                                            float lt, MarchAux& aux, float3 sun, float3 sunInv) {
  using M = MarchGroup<GL>;
  if (R.channel != DCG_RENDER_FLUID || lt == 0.f) return lt;
  float dNear, dFar;
  if (!rayDomain(P, dNear, dFar, origin, sunInv)) return lt;
  float3 pos = origin;
  if (dNear > 0.f) {
    pos = v3add(pos, v3mul(sun, dNear));
    dFar = dFar - dNear;
  }
  const float step = fmaxf(dFar / 100.f, 1e-1f);
  const float3 ds = v3mul(sun, step);
  float density = 0.f;
  if constexpr (GL == 1) {
    for (float d = step; d < dFar && density < 5.f; d = d + step) {
      pos = v3add(pos, ds);
      smp.template sample<GL>(P, R.precise, pos, aux);
      density = density + aux.density * P.dx * step;
    }
    return lt * marchExp(-density);
  }
  // the lane's step of the first round: distance and position after lane() + 1 steps
  const int lane = M::lane();
  float d = step;
  pos = v3add(pos, ds);
#pragma unroll
  for (int j = 1; j < GL; j++) {
    const float3 q = v3add(pos, ds);
    if (lane >= j) {
      pos = q;
      d = d + step;
    }
  }
  for (;;) {
    float c = 0.f;  // adds nothing for a lane past the end
    if (d < dFar) {
      smp.template sample<GL>(P, R.precise, pos, aux);
      c = aux.density * P.dx * step;
    }
    M::each([&](auto J) {
      const float cj = M::template from<decltype(J)::value>(c);
      density = density < 5.f ? density + cj : density;
    });
    if (!(M::template from<GL - 1>(d) < dFar) || !(density < 5.f)) break;
#pragma unroll
    for (int j = 0; j < GL; j++) {
      pos = v3add(pos, ds);
      d = d + step;
    }
  }
  return lt * marchExp(-density);
}

// What a ray meets behind the fluid (src/raymarching.cuh:144-186), with the solid scene's part of
// the light there.
enum : int { MARCH_NONE, MARCH_SCENE, MARCH_FLOOR, MARCH_DEBUG };
struct MarchSolid {
  float d;
  int what;
  float lt;
};
__device__ __forceinline__ MarchSolid marchSolid(const dcg_params& P, const dcg_render_params& R, float3 origin, float3 dir,
                                                 float3 sun) {
  const float sliceZ = (float)P.gz * .5f;
  MarchSolid m{FLT_MAX, MARCH_NONE, 1.f};
  if (R.channel != DCG_RENDER_FLUID && (sliceZ - origin.z) * dir.z > 0.f) {
    const float dDebug = (sliceZ - origin.z) / dir.z;
    const float dx = origin.x + dDebug * dir.x, dy = origin.y + dDebug * dir.y;
    if (dx >= 0.f && dy >= 0.f && dx < (float)P.gx && dy < (float)P.gy && dDebug < m.d) {
      m.d = dDebug;
      m.what = MARCH_DEBUG;
    }
  }
  if (R.solids && (0.f - origin.y) * dir.y > 0.f) {
    const float dFloor = (0.f - origin.y) / dir.y;
    if (dFloor < m.d) {
      m.d = dFloor;
      m.what = MARCH_FLOOR;
    }
  }
  if (R.solids && P.enable_additional_solids) {
    float sdf = FLT_MAX, dScene = 0.f;
    for (int i = 0; i < 100; i++) {
      sdf = sceneSDF(P, v3add(origin, v3mul(dir, dScene)));
      if (sdf < 1e-1f || dScene >= m.d) break;
      dScene = dScene + sdf;
    }
    if (sdf < 1e-1f && dScene < m.d) {
      m.d = dScene;
      m.what = MARCH_SCENE;
    }
    if (R.shadows && (m.what == MARCH_SCENE || m.what == MARCH_FLOOR)) {
      float3 pos = v3add(origin, v3mul(dir, m.d));
      if (m.what == MARCH_FLOOR) pos.y = 0.f;
      m.lt = sceneLight(P, R, pos, sun);
    }
  }
  return m;
}

// Where a ray that enters the domain at dNear begins its march (Z_NEAR 10).
__device__ __forceinline__ float marchStart(float dNear) { return fmaxf(0.f, fmaxf(dNear, 10.f)); }

// raymarch (src/raymarching.cuh:123-275); returns (color, alpha), the same in the whole group.
template <int GL, class S>
__device__ __forceinline__ float4 rayMarch(const S& smp, const dcg_params& P, const dcg_render_params& R, float3 origin,
                                           float3 dir, float3 sun, const MarchSolid& solid) {
  using M = MarchGroup<GL>;
  const float ambientInv = 1.f - R.ambient;
  const float floorIllum = fmaxf(0.f, sun.y);
  const float sliceZ = (float)P.gz * .5f;
  const float3 dirInv = make_float3(1.f / dir.x, 1.f / dir.y, 1.f / dir.z);
  const float3 sunInv = make_float3(1.f / sun.x, 1.f / sun.y, 1.f / sun.z);
  float3 color = make_float3(0.f, 0.f, 0.f);
  float alpha = 0.f, illum;
  MarchAux aux;
  aux.ipos = make_int3(0, 0, 0);
  aux.frac = make_float3(0.f, 0.f, 0.f);
  aux.density = 0.f;
#pragma unroll
  for (int k = 0; k < 8; k++) aux.cell[k] = 0;
  const float dSolid = solid.d;
  const int what = solid.what;
  if (R.channel == DCG_RENDER_FLUID) {
    float dNear, dFar;
    if (rayDomain(P, dNear, dFar, origin, dirInv)) {
      float dCurrent = marchStart(dNear);
      const float dMax = fminf(dFar, dSolid);
      auto shade = [&](float light, float sa) {
        light = R.ambient + light * ambientInv;
        marchMix(make_float3(light * R.smoke_color[0], light * R.smoke_color[1], light * R.smoke_color[2]), sa, color, alpha);
      };
      auto next = [&](float d) { return fminf(fmaxf(d * 1.f, d + .5f), dMax); };  // STEP_MULTIPLIER 1
      float3 pos = v3add(origin, v3mul(dir, dCurrent));
      while (GL == 1 && dCurrent < dMax && alpha <= .99f) {
        const float3 prev = pos;
        dCurrent = next(dCurrent);
        pos = v3add(origin, v3mul(dir, dCurrent));
        const float3 mid = v3mul(v3add(prev, pos), .5f);
        smp.template sample<GL>(P, R.precise, mid, aux);
        if (!(aux.density > 1e-6f)) continue;
        const float sa = densityToAlpha(P, aux.density, v3len(v3sub(pos, prev)));
        shade(R.shadows ? fluidLight<GL>(smp, P, R, mid, sceneLight(P, R, mid, sun), aux, sun, sunInv) : 1.f, sa);
      }
      const int lane = M::lane();
      while (GL > 1 && dCurrent < dMax && alpha <= .99f) {
        // the next GL steps: lane k goes from the distance after k of them to the one after k + 1
        float d0 = dCurrent;
#pragma unroll
        for (int j = 1; j <= GL; j++) {
          dCurrent = next(dCurrent);
          if (j < GL && lane >= j) d0 = dCurrent;
        }
        float density = 0.f, sa = 0.f, lt = 1.f;
        float3 mid = make_float3(0.f, 0.f, 0.f);
        if (d0 < dMax) {
          const float3 prev = v3add(origin, v3mul(dir, d0));
          pos = v3add(origin, v3mul(dir, next(d0)));
          mid = v3mul(v3add(prev, pos), .5f);
          smp.template sample<GL>(P, R.precise, mid, aux);
          density = aux.density;
          if (density > 1e-6f) {
            sa = densityToAlpha(P, density, v3len(v3sub(pos, prev)));
            if (R.shadows) lt = sceneLight(P, R, mid, sun);
          }
        }
        // the steps that meet fluid, in order
        for (uint32_t todo = M::ballot(density > 1e-6f); todo != 0 && alpha <= .99f; todo &= todo - 1) {
          const int j = __ffs(todo) - 1;
          const float saj = M::at(sa, j);
          float light = 1.f;
          if (R.shadows) {
            const float3 mj = make_float3(M::at(mid.x, j), M::at(mid.y, j), M::at(mid.z, j));
            light = fluidLight<GL>(smp, P, R, mj, M::at(lt, j), aux, sun, sunInv);
          }
          shade(light, saj);
        }
      }
    }
  }
  float3 pos = v3add(origin, v3mul(dir, dSolid));
  const float bgAlpha = densityToAlpha(P, 1e-6f, dSolid);
  if (what == MARCH_SCENE) {
    const float3 n = sceneNormal(P, pos);
    illum = fmaxf(0.f, n.x * sun.x + n.y * sun.y + n.z * sun.z);
    if (R.shadows) illum = illum * fluidLight<GL>(smp, P, R, pos, solid.lt, aux, sun, sunInv);
    illum = R.ambient + illum * ambientInv;
    marchMix(make_float3(illum * R.scene_color[0], illum * R.scene_color[1], illum * R.scene_color[2]), 1.f - bgAlpha,
             color, alpha);
  }
  if (what == MARCH_FLOOR) {
    pos.y = 0.f;
    illum = floorIllum;
    if (R.shadows) illum = illum * fluidLight<GL>(smp, P, R, pos, solid.lt, aux, sun, sunInv);
    illum = R.ambient + illum * ambientInv;
    illum = illum * (1.f + .1f * fmodf(fabsf(floorf(pos.x / (float)P.gx) + floorf(pos.z / (float)P.gx)), 2.f));
    marchMix(make_float3(illum * R.floor_color[0], illum * R.floor_color[1], illum * R.floor_color[2]), 1.f - bgAlpha,
             color, alpha);
  }
  if (what == MARCH_DEBUG) {
    pos.z = sliceZ;
    smp.template sample<GL>(P, R.precise, pos, aux);
    if (R.channel == DCG_RENDER_DENSITY) {
      const float v = aux.density * 1e2f;
      marchMix(make_float3(v, 0.f, 0.f), 1.f, color, alpha);
    }
    if (R.channel == DCG_RENDER_VELOCITY) {
      const float v = v3len(smp.velocity(aux)) * 1e-1f;
      marchMix(make_float3(v - 2.f, v - 1.f, v), 1.f, color, alpha);
    }
    if (R.channel == DCG_RENDER_RESOLUTION) {
      const float c = (float)((aux.ipos.x / 4 + aux.ipos.y / 4) % 2);
      marchMix(make_float3(c, c, c), 1.f, color, alpha);
    }
    if (R.channel == DCG_RENDER_FLUIDITY) {
      const float f = smp.fluidity(aux);
      marchMix(make_float3(f, f, f), 1.f, color, alpha);
    }
  }
  return make_float4(color.x, color.y, color.z, alpha);
}

// The camera ray of pixel (x, y) offset by (dx, dy).
__device__ __forceinline__ float3 marchDirection(const dcg_render_params& R, int x, int y, float dx, float dy) {
  const float cx = .5f * (float)R.width, cy = .5f * (float)R.height;
  const float s = R.fov / fmaxf(cx, cy);
  const float3 view = v3norm(make_float3(((float)x + dx - cx) * s, ((float)y + dy - cy) * s, 1.f));
  return make_float3(view.x, view.z * R.eye_dir[1] - view.y * R.eye_dir[2], view.y * R.eye_dir[1] + view.z * R.eye_dir[2]);
}
__device__ __forceinline__ float3 marchOrigin(const dcg_params& P, const dcg_render_params& R) {
  return make_float3(R.eye_origin[0] * P.rdx, R.eye_origin[1] * P.rdx, R.eye_origin[2] * P.rdx);
}

// For rays that meet no fluid.
struct NoFluid {
  template <int GL>
  __device__ void sample(const dcg_params&, int, float3, MarchAux&) const {}
  __device__ float3 velocity(const MarchAux&) const { return make_float3(0.f, 0.f, 0.f); }
  __device__ float fluidity(const MarchAux&) const { return 0.f; }
};
// A thread per ray before the rays are marched by several lanes each (one ray per pixel, the marched
// channel): a ray that has no fluid to cross and whose background no fluid can shade is finished here;
// of the others the image takes what they meet behind the fluid: d, what, lt, and kMarchOpen (a NaN that
// no arithmetic makes) where a finished pixel has its opacity.
static constexpr int kMarchOpen = 0x7FC5A5A5;
static __global__ void __launch_bounds__(256) k_render_begin(dcg_params P, dcg_render_params R, float4* __restrict__ out) {
  const int x = blockIdx.x * 16 + (int)(threadIdx.x % 16), y = blockIdx.y * 16 + (int)(threadIdx.x / 16);
  if (x >= R.width || y >= R.height) return;
  const float3 sun = make_float3(R.sun_dir[0], R.sun_dir[1], R.sun_dir[2]);
  const float3 origin = marchOrigin(P, R), dir = marchDirection(R, x, y, 0.f, 0.f);
  const MarchSolid m = marchSolid(P, R, origin, dir, sun);
  float dNear, dFar;
  bool open = rayDomain(P, dNear, dFar, origin, make_float3(1.f / dir.x, 1.f / dir.y, 1.f / dir.z)) &&
              marchStart(dNear) < fminf(dFar, m.d);
  if (!open && R.shadows && m.what != MARCH_NONE && m.lt != 0.f) {
    float3 pos = v3add(origin, v3mul(dir, m.d));
    if (m.what == MARCH_FLOOR) pos.y = 0.f;
    open = rayDomain(P, dNear, dFar, pos, make_float3(1.f / sun.x, 1.f / sun.y, 1.f / sun.z));
  }
  float4 c = make_float4(m.d, __int_as_float(m.what), m.lt, __int_as_float(kMarchOpen));
  if (!open) {
    c = rayMarch<1>(NoFluid{}, P, R, origin, dir, sun, m);
    c = make_float4(0.f + c.x, 0.f + c.y, 0.f + c.z, 0.f + c.w);  // k_render's sum over one ray
  }
  out[(size_t)y * R.width + x] = c;
}

// k_dcgrid_render / k_uniform_render: per pixel, aa_samples^2 rays averaged. A workgroup takes a
// tile of T x T pixels with GL lanes per ray. BEGUN: the pixel's entry of the image comes from
// k_render_begin. One lane per ray runs on images that fill the chip: four wavefronts a SIMD (at most 128
// VGPRs) instead of three take 1.05-1.16x off them.
template <int GL, int T, bool BEGUN, class S>
__global__ void __launch_bounds__(T* T* GL, GL == 1 ? 4 : 1) k_render(S smp, dcg_params P, dcg_render_params R, float4* __restrict__ out) {
  const int ray = (int)(threadIdx.x / GL);
  const int x = blockIdx.x * T + ray % T, y = blockIdx.y * T + ray / T;
  if (x >= R.width || y >= R.height) return;
  const float step = 1.f / R.aa_samples;
  const float3 origin = marchOrigin(P, R);
  const float3 sun = make_float3(R.sun_dir[0], R.sun_dir[1], R.sun_dir[2]);
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (float dx = 0.f; dx < 1.f; dx = dx + step)
    for (float dy = 0.f; dy < 1.f; dy = dy + step) {
      const float3 dir = marchDirection(R, x, y, dx, dy);
      MarchSolid solid;
      if (BEGUN) {
        const float4 m = out[(size_t)y * R.width + x];
        if (__float_as_int(m.w) != kMarchOpen) return;  // finished there
        solid = MarchSolid{m.x, __float_as_int(m.y), m.z};
      } else {
        solid = marchSolid(P, R, origin, dir, sun);
      }
      const float4 c = rayMarch<GL>(smp, P, R, origin, dir, sun, solid);
      acc = make_float4(acc.x + c.x, acc.y + c.y, acc.z + c.z, acc.w + c.w);
    }
  if (MarchGroup<GL>::lane() != 0) return;
  const float w = step * step;
  out[(size_t)y * R.width + x] = make_float4(acc.x * w, acc.y * w, acc.z * w, acc.w * w);
}

// The launches of a render: lanes per ray, and whether k_render_begin goes first.
//
// The ray's fixed cost and the sums in its order are paid by every lane, so lanes win while the image
// has too few rays for the chip (2^18 threads of this kernel are resident) or rays of very unequal
// length (shadow marches), and lose where a thread per ray fills it. The lines lie where no scene with fluid
// in view is slower than with one lane by more than the noise (MI355X; DCGrid scenes of 128^3 to 512^3 cells,
// plume and sphere, and dense grids, 64^3 with a plume and 200^3 filled with fluid; gain over one lane):
//   DCGrid, shadows      724 x 724: 16 lanes 5.1-8.3x, 4 lanes 3.0-4.1x; 1920 x 1080: 4 lanes 1.5-2.1x, 16
//                        1.0-2.0x; 3840 x 2160: 4 lanes 0.8-1.1x
//   DCGrid, no shadows   512 x 512: 16 and 4 lanes 1.6-2.5x; 1024 x 768: 4 lanes 1.05-1.45x; 1920 x 1080: 0.8-1.0x
//   dense, shadows       256 x 256: 16 lanes 4.2-4.7x; 512 x 512: 4 lanes 1.6-2.6x, 16 1.3-3.2x; 1024 x 768: 4 lanes
//                        1.3-1.9x, 16 0.75-1.4x; 1920 x 1080: 4 lanes 0.8-1.2x
//   dense, no shadows    128 x 128: 16 lanes 2.8-3.8x; 256 x 256: 4 lanes 2.0x, 16 1.3-1.8x; 512 x 512: 4 lanes
//                        1.0-1.2x; 724 x 724: 0.9-1.0x
// A solid scene's traces (up to 200 scene distances a ray) cannot be shared by a ray's lanes and are left to
// k_render_begin, a thread per ray. With a terrain, each distance a 5-octave noise, they are most of
// the image and no longer hidden beside the march: 16 lanes up to 512 x 512 (there 1.2-1.9x; 0.95 with coarse
// samples or no fluid in view), one above (0.8-1.1 with 16), and one with several rays per pixel, which the
// image cannot hold (16 lanes 0.1-0.5x). The finishing of rays that meet no fluid is worth a launch of its own from
// 2^16 pixels on; an image of nothing but such rays pays for it (1920 x 1080: 21 -> 65 us).
struct MarchRoute {
  int lanes;
  bool begin;
};
template <class S>
MarchRoute marchRoute(const dcg_params& P, const dcg_render_params& R) {
  if (R.channel != DCG_RENDER_FLUID) return {1, false};  // one sample per ray
  const size_t pixels = (size_t)R.width * R.height;
  const bool scene = R.solids && P.enable_additional_solids, single = R.aa_samples <= 1.f;
  int lanes;
  if (scene && P.solid_mode == DCG_SOLID_TERRAIN) {
    lanes = single && pixels <= (size_t)1 << 18 ? 16 : 1;
  } else {
    const int most16 = S::kDense ? (R.shadows ? 17 : 15) : (R.shadows ? 19 : 18);  // log2 of the pixels
    const int most4 = S::kDense ? (R.shadows ? 20 : 18) : (R.shadows ? 21 : 20);
    lanes = pixels <= (size_t)1 << most16 ? 16 : pixels <= (size_t)1 << most4 ? 4 : 1;
  }
  return {lanes, lanes > 1 && single && (scene || pixels > (size_t)1 << 16)};
}
static inline dim3 marchGrid(const dcg_render_params& R, int tile) {
  return dim3((unsigned)((R.width + tile - 1) / tile), (unsigned)((R.height + tile - 1) / tile));
}
static inline void launchRenderBegin(const dcg_params& P, const dcg_render_params& R, float4* out, hipStream_t stream) {
  k_render_begin<<<marchGrid(R, 16), 256, 0, stream>>>(P, R, out);
}
template <class S>
void launchRender(const S& smp, MarchRoute route, const dcg_params& P, const dcg_render_params& R, float4* out,
                  hipStream_t stream) {
  if (route.lanes == 1)
    k_render<1, 16, false><<<marchGrid(R, 16), 256, 0, stream>>>(smp, P, R, out);
  else if (route.lanes == 4 && route.begin)
    k_render<4, 8, true><<<marchGrid(R, 8), 256, 0, stream>>>(smp, P, R, out);
  else if (route.lanes == 4)
    k_render<4, 8, false><<<marchGrid(R, 8), 256, 0, stream>>>(smp, P, R, out);
  else if (route.begin)
    k_render<16, 4, true><<<marchGrid(R, 4), 256, 0, stream>>>(smp, P, R, out);
  else
    k_render<16, 4, false><<<marchGrid(R, 4), 256, 0, stream>>>(smp, P, R, out);
}

}  // namespace dcg
