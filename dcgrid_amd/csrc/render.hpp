// render.hpp — gfx950 ray marcher over the simulation fields: FluidSimulation::render
// (src/fluid_simulation.h:19) for both grids, following src/raymarching.cuh:63-275 with the
// samplers of src/dcgrid/dcgrid_rendering.cu:6-64 and src/uniformgrid/uniformgrid_rendering.cu:5-47.
//
// Sixteen lanes per ray (MarchGroup). Every float operation is written out in the order of the
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
// GL = 1 is the plain loop, for the debug slices (one sample per ray, nothing to share).
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
  // the lane's step of the first round: distance and position after lane() + 1 steps
  const int lane = M::lane();
  float d = step;
  pos = v3add(pos, ds);
  if (GL > 1) {
#pragma unroll
    for (int j = 1; j < GL; j++) {
      const float3 q = v3add(pos, ds);
      if (lane >= j) {
        pos = q;
        d = d + step;
      }
    }
  }
  float density = 0.f;
  for (;;) {
    float c = 0.f;  // adds nothing for a lane past the end
    if (d < dFar) {
      smp.sample(P, R.precise, pos, aux);
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
      float dCurrent = fmaxf(0.f, fmaxf(dNear, 10.f));  // Z_NEAR
      const float dMax = fminf(dFar, dSolid);
      const int lane = M::lane();
      auto next = [&](float d) { return fminf(fmaxf(d * 1.f, d + .5f), dMax); };  // STEP_MULTIPLIER 1
      while (dCurrent < dMax && alpha <= .99f) {
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
          const float3 prev = v3add(origin, v3mul(dir, d0)), pos = v3add(origin, v3mul(dir, next(d0)));
          mid = v3mul(v3add(prev, pos), .5f);
          smp.sample(P, R.precise, mid, aux);
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
          illum = 1.f;
          if (R.shadows) {
            const float3 mj = make_float3(M::at(mid.x, j), M::at(mid.y, j), M::at(mid.z, j));
            illum = illum * fluidLight<GL>(smp, P, R, mj, M::at(lt, j), aux, sun, sunInv);
          }
          illum = R.ambient + illum * ambientInv;
          marchMix(make_float3(illum * R.smoke_color[0], illum * R.smoke_color[1], illum * R.smoke_color[2]), saj, color,
                   alpha);
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
    smp.sample(P, R.precise, pos, aux);
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

// What every pixel's ray meets behind the fluid, left in the image for k_render (one ray per
// pixel): d, what and lt in x, y and z.
static __global__ void __launch_bounds__(256) k_render_solids(dcg_params P, dcg_render_params R, float4* __restrict__ out) {
  const int x = blockIdx.x * 16 + (int)(threadIdx.x % 16), y = blockIdx.y * 16 + (int)(threadIdx.x / 16);
  if (x >= R.width || y >= R.height) return;
  const float3 sun = make_float3(R.sun_dir[0], R.sun_dir[1], R.sun_dir[2]);
  const MarchSolid m = marchSolid(P, R, marchOrigin(P, R), marchDirection(R, x, y, 0.f, 0.f), sun);
  out[(size_t)y * R.width + x] = make_float4(m.d, __int_as_float(m.what), m.lt, 0.f);
}

// k_dcgrid_render / k_uniform_render: per pixel, aa_samples^2 rays averaged. A workgroup takes a
// tile of T x T pixels with GL lanes per ray. SOLIDS: the pixel's entry of the image holds what its
// one ray meets behind the fluid (k_render_solids).
template <int GL, int T, bool SOLIDS, class S>
__global__ void __launch_bounds__(T* T* GL) k_render(S smp, dcg_params P, dcg_render_params R, float4* __restrict__ out) {
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
      if (SOLIDS) {
        const float4 m = out[(size_t)y * R.width + x];
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

// The launches of a render. The marched channel takes 16 lanes per ray up to 512 K pixels and 4 above,
// the debug slices one thread. The ray's fixed cost is paid by every lane, so once the image alone
// fills the chip fewer lanes win (1920 x 1080, 16 -> 4 lanes: plume 24.1 -> 16.5 ms, dense grid 2.9 ->
// 1.1 ms, terrain 15.2 -> 11.1 ms; at 512 x 512 16 lanes are the faster, 8.5 -> 4.4 ms on the plume).
// A solid scene's sphere traces (up to 200 scene distances a ray, each a 5-octave noise with a
// terrain) cannot be shared by a ray's lanes: a pass of its own takes them a thread per ray, and
// leaves its results in the image, which holds them for one ray per pixel; with several the whole
// march runs a thread per ray (a trace by 16 lanes alike takes 16 times the instructions: a terrain
// image of 1024 x 768 took 17.8 ms with the traces in the march's workgroups, 4.4 ms this way).
template <class S>
void launchRender(const S& smp, const dcg_params& P, const dcg_render_params& R, float4* out, hipStream_t stream) {
  auto grid = [&](int t) { return dim3((unsigned)((R.width + t - 1) / t), (unsigned)((R.height + t - 1) / t)); };
  const bool scene = R.solids && P.enable_additional_solids;
  const bool wide = (size_t)R.width * R.height <= (size_t)512 * 1024;
  if (R.channel != DCG_RENDER_FLUID || (scene && R.aa_samples > 1.f)) {
    k_render<1, 16, false><<<grid(16), 256, 0, stream>>>(smp, P, R, out);
  } else if (scene) {
    k_render_solids<<<grid(16), 256, 0, stream>>>(P, R, out);
    if (wide)
      k_render<16, 4, true><<<grid(4), 256, 0, stream>>>(smp, P, R, out);
    else
      k_render<4, 8, true><<<grid(8), 256, 0, stream>>>(smp, P, R, out);
  } else if (wide) {
    k_render<16, 4, false><<<grid(4), 256, 0, stream>>>(smp, P, R, out);
  } else {
    k_render<4, 8, false><<<grid(8), 256, 0, stream>>>(smp, P, R, out);
  }
}

}  // namespace dcg
