// tc_adjoint.hip -- reverse-mode derivative of hit distance with respect to
// height-map texels (no reference counterpart).
//
// Forward chain per ray, with the tessellation pattern and the hit triangle
// frozen: texels -> bilinear height H(u_k, v_k) at each of the hit
// triangle's three generated vertices -> P_k = base_k + normal_k *
// (heightScale_k * H + heightOffset_k) -> t, the distance along the ray to
// the plane through P_0, P_1, P_2.  Differentiating o + t d = sum_k b_k P_k
// (sum b_k = 1) along the plane normal n gives dt/dP_k = b_k n / (n . d).
// The chain is evaluated in object space, where t equals the world-space
// distance because the direction is carried over linearly.
#include <algorithm>

#include "tc_device.h"

namespace tc {

int num_cu_public();

// A workgroup takes RAYS consecutive rays.  Rays that are neighbours move the
// same texels: with one global atomic per contribution (12 a ray), the launch
// waited for same-word atomics (384^2 rays on 64 x 64 quads, every texel
// receiving about 100 adds: 141 us; 512^2 rays on their tessellation: 57 us).  So
// a workgroup sums its contributions in an LDS table of kAdjointSlots slots a ray
// keyed by the texel's address (open addressing, kAdjointProbes slots tried) and
// adds each entry to memory once: 28 us both.  Neighbouring texels take
// neighbouring slots; a multiplicative hash over half the slots took 34 and 52
// us.  What finds no slot (scattered rays) goes to memory at once.
constexpr uint32_t kAdjointSlots = 4;  // 48 bytes a ray
constexpr uint32_t kAdjointProbes = 4;

template <uint32_t SLOTS>
__device__ __forceinline__ void add_texel(uint64_t* keys, float* sums, float* texel, float v) {
  const uint64_t key = reinterpret_cast<uint64_t>(texel);
  // neighbouring texels take neighbouring slots (LDS banks)
  uint32_t s = ((uint32_t)(key >> 2) + (uint32_t)(key >> 14) * 619u) & (SLOTS - 1);
  for (uint32_t probe = 0; probe < kAdjointProbes; probe++, s = (s + 1) & (SLOTS - 1)) {
    uint64_t held = __hip_atomic_load(keys + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (held == 0) {
      if (__hip_atomic_compare_exchange_strong(keys + s, &held, key, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP))
        held = key;
    }
    if (held == key) {
      unsafeAtomicAdd(sums + s, v);
      return;
    }
  }
  unsafeAtomicAdd(texel, v);
}

template <uint32_t SLOTS>
__device__ __forceinline__ void adjoint_ray(const tc_adjoint_params& p, uint32_t r, uint64_t* keys, float* sums) {
  const float g = p.gradT[r];
  if (g == 0.0f) return;
  const tc_hit h = p.hits[r];
  if (!(h.t >= 0.0f) || h.instanceID == 0xFFFFFFFFu) return;
  const uint4 hv = reinterpret_cast<const uint4*>(p.hitVertices)[r];
  if (hv.x == 0xFFFFFFFFu) return;
  const float* m = p.tlasInstances[h.instanceID].worldToObject;
  const tc_ray ray = p.rays[r];
  const v3 d = mk((m[0] * ray.direction[0] + m[1] * ray.direction[1]) + m[2] * ray.direction[2],
                  (m[4] * ray.direction[0] + m[5] * ray.direction[1]) + m[6] * ray.direction[2],
                  (m[8] * ray.direction[0] + m[9] * ray.direction[1]) + m[10] * ray.direction[2]);
  const uint32_t vi[3] = {hv.x, hv.y, hv.z};
  const uint64_t gv = reinterpret_cast<uint64_t>(p.genVertices);
  const v3 p0 = ld3(gv, vi[0]), p1 = ld3(gv, vi[1]), p2 = ld3(gv, vi[2]);
  const v3 n = cross(sub(p1, p0), sub(p2, p0));
  const float nd = dot(n, d);
  if (nd == 0.0f) return;
  const float b[3] = {(1.0f - h.u) - h.v, h.u, h.v};
  const float gs = g / nd;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float4* tp = reinterpret_cast<const float4*>(p.tape + vi[k]);
    const float4 q0 = tp[0], q1 = tp[1], q2 = tp[2];
    const uint32_t tex = __float_as_uint(q2.z);
    if (tex >= p.numTextures) continue;
    float* grad = p.gradTexels[tex];
    if (!grad) continue;
    const v3 nk = mk(q0.w, q1.x, q1.y);
    const float coef = ((gs * b[k]) * q2.x) * dot(n, nk);
    if (coef == 0.0f) continue;
    const tc_displacement_texture t = p.textures[tex];
    uint64_t idx[4];
    float w[4];
    bilinear_footprint(t.width, t.height, q1.z, q1.w, idx, w);
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (w[j] != 0.0f) add_texel<SLOTS>(keys, sums, grad + idx[j], coef * w[j]);
  }
}

template <uint32_t RAYS>
__global__ __launch_bounds__(RAYS) void k_depth_adjoint(tc_adjoint_params p) {
  constexpr uint32_t SLOTS = kAdjointSlots * RAYS;
  __shared__ uint64_t s_key[SLOTS];  // texel address, 0: free
  __shared__ float s_sum[SLOTS];
  for (uint64_t base = blockIdx.x * (uint64_t)RAYS; base < p.numRays; base += gridDim.x * (uint64_t)RAYS) {
    for (uint32_t i = threadIdx.x; i < SLOTS; i += RAYS) s_key[i] = 0, s_sum[i] = 0.0f;
    __syncthreads();
    if (threadIdx.x < p.numRays - base) adjoint_ray<SLOTS>(p, (uint32_t)base + threadIdx.x, s_key, s_sum);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < SLOTS; i += RAYS)
      if (s_key[i]) unsafeAtomicAdd(reinterpret_cast<float*>(s_key[i]), s_sum[i]);
    __syncthreads();
  }
}

// The largest workgroup that leaves half of the CUs with one, from 1024 rays
// down to 128: the adds to a CU's table follow one another, 17 us for 1024 rays
// however few workgroups there are.  Workgroups of 1024 / 512 / 256 / 128 and
// plain atomics (row order, 64 x 64 quads, map 512^2): 64^2 rays 19.0 / 12.2 / 9.2 /
// 7.8 and 6.9 us, 128^2 20.5 / 14.3 / 11.4 / 10.0 and 8.6, 193^2 22.8 / 16.8 / 16.3 /
// 15.9 and 15.8, 256^2 22.4 / 14.8 / 15.9 / 17.1 and 17.8, 384^2 24.7 / 27.7 / 26.5 /
// 30.9 and 33.5; on 8 x 8 quads, every texel moved by hundreds of rays, 64^2 26.3 /
// 16.4 / 10.2 / 9.0 and 30.3, 256^2 28.0 / 17.6 / 12.1 / 14.5 and 339.
static uint32_t adjoint_rays(uint32_t numRays) {
  uint32_t r = 1024;
  while (r > 128 && numRays < (uint64_t)r * num_cu_public() / 2) r /= 2;
  return r;
}

template <uint32_t RAYS>
static void launch_adjoint(const tc_adjoint_params& p, hipStream_t stream) {
  const uint32_t grid = std::min<uint32_t>((p.numRays - 1) / RAYS + 1, (uint32_t)num_cu_public() * 8);
  hipLaunchKernelGGL(k_depth_adjoint<RAYS>, dim3(grid), dim3(RAYS), 0, stream, p);
}

}  // namespace tc

using namespace tc;

extern "C" tc_status tc_depth_adjoint(const tc_adjoint_params* p, tc_stream stream) {
  if (!p) return TC_ERROR_INVALID_ARGUMENT;
  if (p->numRays == 0) return TC_OK;
  if (!p->rays || !p->hits || !p->hitVertices || !p->gradT || !p->genVertices || !p->tape || !p->tlasInstances ||
      (p->numTextures && (!p->textures || !p->gradTexels)))
    return TC_ERROR_INVALID_ARGUMENT;
  switch (adjoint_rays(p->numRays)) {
    case 128: launch_adjoint<128>(*p, (hipStream_t)stream); break;
    case 256: launch_adjoint<256>(*p, (hipStream_t)stream); break;
    case 512: launch_adjoint<512>(*p, (hipStream_t)stream); break;
    default: launch_adjoint<1024>(*p, (hipStream_t)stream); break;
  }
  return hipGetLastError() == hipSuccess ? TC_OK : TC_ERROR_LAUNCH;
}
