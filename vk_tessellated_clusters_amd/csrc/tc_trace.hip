// tc_trace.hip -- primary / shadow ray traversal and the closest-hit decode.
//
// Stands for vkCmdTraceRaysKHR with render_raytrace.rgen.glsl:52-86 (rays),
// the hardware traversal of the cluster BVH, render_raytrace_clusters.rchit.
// glsl:128-236, 338-339 (decode, depth) and render_shading.glsl:263-274
// (shadow rays).  One ray per lane over the four-wide views of the TLAS and
// the BLAS; the lane's stack (LDS, overflowing into private memory) holds
// TLAS and BLAS entries (those of the instance being walked lie above a
// sentinel).  Triangles use the watertight test of
// Woop, Benthin and Wald (JCGT 2013) with an FP64 recomputation of zero edge
// functions; closest-hit ties are broken by (instance, cluster, primitive)
// so the result does not depend on traversal order.
#include <algorithm>

#include "tc_trace.h"

namespace tc {


struct WoopRay {
  float o[3], d[3], inv[3];
  int kx, ky, kz;
  float Sx, Sy, Sz;
};

// (x, y, z)[k] for a lane-varying k in {0, 1, 2} as two selects of
// registers (a dynamic index into an array would go through private memory)
__device__ __forceinline__ float pick3(float x, float y, float z, int k) { return k == 0 ? x : (k == 1 ? y : z); }

// The parts of a ray that box tests read.
__device__ __forceinline__ void setup_box_ray(WoopRay& r, const float o[3], const float dir[3]) {
  for (int k = 0; k < 3; k++) {
    float d = dir[k];
    asm volatile("" : "+v"(d));  // register values: the picks of setup_ray stay selects
    r.o[k] = o[k], r.d[k] = d, r.inv[k] = 1.0f / d;
  }
}

// Whether (plane - o) * inv is a number for every plane, infinite ones
// included: no axis is parallel to the ray and the origin is finite.
__device__ __forceinline__ bool regular_ray(const WoopRay& r) {
  bool ok = true;
  for (int k = 0; k < 3; k++) {
    const float i = fabsf(r.inv[k]);
    ok = ok && i > 0.0f && i < INFINITY && fabsf(r.o[k]) < INFINITY;
  }
  return ok;
}

__device__ __forceinline__ void setup_ray(WoopRay& r, const float o[3], const float dir[3]) {
  setup_box_ray(r, o, dir);
  const float ax = fabsf(r.d[0]), ay = fabsf(r.d[1]), az = fabsf(r.d[2]);
  r.kz = (ax > ay) ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
  r.kx = r.kz == 2 ? 0 : r.kz + 1;
  r.ky = r.kx == 2 ? 0 : r.kx + 1;
  const float dz = pick3(r.d[0], r.d[1], r.d[2], r.kz);
  if (dz < 0.0f) {
    const int t = r.kx;
    r.kx = r.ky;
    r.ky = t;
  }
  r.Sx = pick3(r.d[0], r.d[1], r.d[2], r.kx) / dz;
  r.Sy = pick3(r.d[0], r.d[1], r.d[2], r.ky) / dz;
  r.Sz = pick3(r.inv[0], r.inv[1], r.inv[2], r.kz);  // 1 / dz
}

// Slab test; returns the entry distance or +inf.  A ray that lies in a plane of
// the box (parallel to it, its origin on it) has 0 * inf in that slab, which
// counts as the other plane's infinity: it misses.
__device__ __forceinline__ float box_hit(const WoopRay& r, const float lo[3], const float hi[3], float tmin, float tmax) {
  float tn = tmin, tf = tmax;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float t0 = (lo[k] - r.o[k]) * r.inv[k];
    const float t1 = (hi[k] - r.o[k]) * r.inv[k];
    tn = fmaxf(tn, fminf(t0, t1));
    tf = fminf(tf, fmaxf(t0, t1));
  }
  return tn <= tf * 1.0000005f ? tn : INFINITY;
}

struct TriDet {
  float t, V, W, det;
};

// Woop et al. 2013 with barycentrics V / det (vertex 1) and W / det
// (vertex 2), which only a ray's closest hit divides out
__device__ __forceinline__ bool tri_test(const WoopRay& r, const float* p0, const float* p1, const float* p2, bool cullBack,
                                         float tmin, float tmax, TriDet& h) {
  const float A0 = p0[0] - r.o[0], A1 = p0[1] - r.o[1], A2 = p0[2] - r.o[2];
  const float B0 = p1[0] - r.o[0], B1 = p1[1] - r.o[1], B2 = p1[2] - r.o[2];
  const float C0 = p2[0] - r.o[0], C1 = p2[1] - r.o[1], C2 = p2[2] - r.o[2];
  const float Akz = pick3(A0, A1, A2, r.kz), Bkz = pick3(B0, B1, B2, r.kz), Ckz = pick3(C0, C1, C2, r.kz);
  const float Ax = pick3(A0, A1, A2, r.kx) - r.Sx * Akz, Ay = pick3(A0, A1, A2, r.ky) - r.Sy * Akz;
  const float Bx = pick3(B0, B1, B2, r.kx) - r.Sx * Bkz, By = pick3(B0, B1, B2, r.ky) - r.Sy * Bkz;
  const float Cx = pick3(C0, C1, C2, r.kx) - r.Sx * Ckz, Cy = pick3(C0, C1, C2, r.ky) - r.Sy * Ckz;
  float U = Cx * By - Cy * Bx;
  float V = Ax * Cy - Ay * Cx;
  float W = Bx * Ay - By * Ax;
  if (U == 0.0f || V == 0.0f || W == 0.0f) {
    U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
    V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
    W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
  }
  if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
  const float det = (U + V) + W;
  if (det == 0.0f) return false;
  if (cullBack && det < 0.0f) return false;
  const float Az = r.Sz * Akz, Bz = r.Sz * Bkz, Cz = r.Sz * Ckz;
  const float T = (U * Az + V * Bz) + W * Cz;
  const float t = T / det;
  if (!(t >= tmin && t <= tmax)) return false;
  h.t = t;
  h.V = V, h.W = W, h.det = det;
  return true;
}

struct HitState {
  tc_hit h;
  const char* clas;  // CLAS block of the best hit
  uint32_t word;     // its triangle word
};

__device__ __forceinline__ bool key_less(float t, uint32_t i, uint32_t c, uint32_t p, const tc_hit& best) {
  if (t != best.t) return t < best.t;
  if (i != best.instanceID) return i < best.instanceID;
  if (c != best.clusterID) return c < best.clusterID;
  return p < best.primitiveID;
}

__device__ __forceinline__ void xform34(const float* m, const float v[3], float w, float out[3]) {
#pragma unroll
  for (int r = 0; r < 3; r++) out[r] = ((m[4 * r] * v[0] + m[4 * r + 1] * v[1]) + m[4 * r + 2] * v[2]) + m[4 * r + 3] * w;
}

__device__ __forceinline__ const float* clas_vertices(const char* clas, uint32_t nt, uint32_t ng) {
  return reinterpret_cast<const float*>(clas + sizeof(tc_clas_header) + ((ng * 24u + 15u) & ~15u) + ((nt * 4u + 15u) & ~15u));
}

// Loads through the global address space: pointers rebuilt from 64-bit
// addresses would otherwise become flat accesses, which also count against
// the LDS counter the stack's ds_* accesses wait on.
template <class T>
__device__ __forceinline__ T gload(const T* p) {
  return *(const __attribute__((address_space(1))) T*)p;
}
// (the HIP vector structs copy through a generic reference: load them as
// native vectors)
__device__ __forceinline__ float4 gload(const float4* p) {
  typedef float v4 __attribute__((ext_vector_type(4)));
  const v4 v = *(const __attribute__((address_space(1))) v4*)p;
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint4 gload(const uint4* p) {
  typedef uint32_t v4 __attribute__((ext_vector_type(4)));
  const v4 v = *(const __attribute__((address_space(1))) v4*)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}

// Slab test of a group box given as six floats; 1 if entered.
__device__ __forceinline__ uint32_t group_hit(const WoopRay& r, float l0, float l1, float l2, float h0, float h1, float h2,
                                              float tmin, float tmax) {
  const float lo[3] = {l0, l1, l2}, hi[3] = {h0, h1, h2};
  return box_hit(r, lo, hi, tmin, tmax) != INFINITY ? 1u : 0u;
}

// Group-box hit mask of the pairs [0, npairs) of a block, P pairs (2P
// boxes) per step with the step's loads issued together; pair p holds
// groups 2p and 2p + 1 in three float4.
template <uint32_t P>
__device__ __forceinline__ uint32_t group_mask(const WoopRay& r, const float4* gq, uint32_t npairs, float tmin, float tmax) {
  uint32_t mask = 0;
  for (uint32_t p0 = 0; p0 < npairs; p0 += P) {
    float4 v[P][3];
    uint32_t pp[P];
#pragma unroll
    for (uint32_t j = 0; j < P; j++) {
      pp[j] = min(p0 + j, npairs - 1);
      v[j][0] = gload(gq + 3 * pp[j]), v[j][1] = gload(gq + 3 * pp[j] + 1), v[j][2] = gload(gq + 3 * pp[j] + 2);
    }
#pragma unroll
    for (uint32_t j = 0; j < P; j++) {
      const float4 a0 = v[j][0], a1 = v[j][1], a2 = v[j][2];
      mask |= group_hit(r, a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, tmin, tmax) << (2 * pp[j]);
      mask |= group_hit(r, a1.z, a1.w, a2.x, a2.y, a2.z, a2.w, tmin, tmax) << (2 * pp[j] + 1);
    }
  }
  return mask;
}

// Intersects one CLAS block, whose header's counts and cluster ID come in
// `info` (tc_accel.blasLeafInfo); updates `best` (closest) or returns true
// on the first hit (any-hit).  The loads of a step are issued together so a
// lane waits for memory once per step rather than once per box or
// triangle: group boxes eight at a time (four 48-byte pairs), then the four
// triangles of each group entered (one 16-byte load of their words, then
// their twelve vertices, issued with the next group's words).  Reads past
// the last group or triangle stay inside the block (its sections are
// rounded up to 16 bytes) or are clamped, and their results are masked off.
__device__ __forceinline__ bool clas_hit(const WoopRay& r, const char* clas, uint64_t info, uint32_t instanceID, bool cullBack,
                                         bool anyHit, float tmin, HitState& best) {
  const uint32_t counts = (uint32_t)info, clusterID = (uint32_t)(info >> 32);
  const uint32_t nt = counts & 0xFF, ng = (counts >> 16) & 0xFF;
  const float4* gq = reinterpret_cast<const float4*>(clas + sizeof(tc_clas_header));
  const uint32_t* tris = reinterpret_cast<const uint32_t*>(clas + sizeof(tc_clas_header) + ((ng * 24u + 15u) & ~15u));
  const float* verts = clas_vertices(clas, nt, ng);
  // group boxes (ng <= 32): eight per step, or two per step when every
  // lane of the wave holds a block of at most two groups (most tessellated
  // parts), which would otherwise test six clamped repeats
  const uint32_t npairs = (ng + 1) >> 1;
  uint32_t mask = __all(npairs <= 1) ? group_mask<1>(r, gq, npairs, tmin, best.h.t)
                                     : group_mask<4>(r, gq, npairs, tmin, best.h.t);
  if (ng < 32) mask &= (1u << ng) - 1u;
  // then the triangles of the groups entered, so the lanes of a wave run
  // the triangle loop together
  if (!mask) return false;
  uint32_t g = __builtin_ctz(mask);
  mask &= mask - 1;
  uint4 w4 = gload(reinterpret_cast<const uint4*>(tris + g * TC_CLAS_GROUP_TRIANGLES));
  while (true) {
    const uint32_t t0 = g * TC_CLAS_GROUP_TRIANGLES;
    uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
    // the next group's words load while this group's vertices do
    const uint32_t gn = mask ? __builtin_ctz(mask) : g;
    w4 = gload(reinterpret_cast<const uint4*>(tris + gn * TC_CLAS_GROUP_TRIANGLES));
    float v[4][9];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (t0 + j >= nt) w[j] = 0;  // vertex 0: an in-bounds read, result unused
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const float* pk = verts + 3 * ((w[j] >> (8 * k)) & 0xFF);
        v[j][3 * k] = gload(pk), v[j][3 * k + 1] = gload(pk + 1), v[j][3 * k + 2] = gload(pk + 2);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (t0 + j >= nt) break;
      TriDet th;
      if (!tri_test(r, v[j], v[j] + 3, v[j] + 6, cullBack, tmin, best.h.t, th)) continue;
      const uint32_t prim = w[j] >> 24;
      if (anyHit) {
        best.h.t = th.t;
        return true;
      }
      if (key_less(th.t, instanceID, clusterID, prim, best.h)) {
        best.h.t = th.t;
        best.h.u = th.V / th.det;
        best.h.v = th.W / th.det;
        best.h.instanceID = instanceID;
        best.h.clusterID = clusterID;
        best.h.primitiveID = prim;
        best.clas = clas;
        best.word = w[j];
      }
    }
    if (!mask) return false;
    g = gn;
    mask &= mask - 1;
  }
}

// Traversal stack of one lane: the first kLdsStack entries in LDS (stride
// 64), the rest in a private array.  TLAS and BLAS entries share it: a kDone
// sentinel lies at its bottom and another below the BLAS entries of the
// instance being walked, so a pop needs no depth test to end a walk.  Bound:
// every visited node pushes at most 3 of its 4 slots, and the four-wide view
// visits every other level, so a ray holds at most 3 * (ceil(dT / 2) +
// ceil(dB / 2)) entries and two sentinels for binary depths dT (TLAS) and dB
// (BLAS).  A Karras tree's depth is at most its distinct key bits plus the
// index bits that break ties.  TLAS keys are a 30-bit Morton code, all ones for
// empty instances (one more bit that differs), above the instance index of at
// most 16 bits; a BLAS covers one instance's segment, whose keys differ only in
// the 24-bit Morton code, and its positions have at most 31 bits (the 32nd marks
// a leaf).
constexpr uint32_t kLdsStack = 16;
constexpr uint32_t kStackDepth = 160;
constexpr uint32_t kTlasDepth = 30 + 1 + 16, kBlasDepth = 24 + 31;
constexpr uint32_t kMostEntries = 3 * ((kTlasDepth + 1) / 2 + (kBlasDepth + 1) / 2);
static_assert(kMostEntries + 2 <= kStackDepth, "entries and sentinels of the deepest trees");
// The node loop hands over to a leaf step when fewer than one in this many of
// the lanes still in their BLAS search (the others hold a leaf): the step costs
// what its leaves cost, so it need not wait for stragglers.  A share, not a
// count, so that the waves of small and of ragged launches, which have few rays,
// do not take their steps with half of them: against fewer than 8 lanes
// icosphere 320 x 180 113 -> 91 us, grid64 480 -> 468, 500 meshes 832 -> 814,
// 3840 x 2160 patches 3730 -> 3697.  1/2 and 1/12 lose at the small images (96
// and 98 us), 1/8 and all at the patches (3750 and 3844).
constexpr uint32_t kSearchShare = 4;
constexpr uint32_t kDone = 0xFFFFFFFFu;

typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(5))) uint32_t private_u32;

// Holds no array itself, so the stack pointer lives in a register; the
// typed pointers make every access a ds_* or scratch_* instruction.  `sp` is
// the byte offset of the next entry as if all of them lay in LDS.
constexpr uint32_t kStackStep = 4 * kWave;
struct RayStack {
  lds_u32* lds;        // this lane's first entry, stride kWave
  private_u32* spill;  // kStackDepth private entries
  uint32_t ldsEnd;     // kLdsStack entries, or 0 with TC_TRACE_PRIVATE_STACK
  uint32_t sp;
  __device__ __forceinline__ lds_u32* entry(uint32_t at) const {
    return (lds_u32*)((__attribute__((address_space(3))) char*)lds + at);
  }
  __device__ __forceinline__ void push(uint32_t e) {
    if (sp < ldsEnd)
      *entry(sp) = e;
    else if (sp < kStackDepth * kStackStep)
      spill[(sp - ldsEnd) / kStackStep] = e;
    sp += kStackStep;
  }
  __device__ __forceinline__ uint32_t pop() {
    sp -= kStackStep;
    return sp < ldsEnd ? *entry(sp) : spill[(sp - ldsEnd) / kStackStep];
  }
};

__device__ __forceinline__ void load_node4(const tc_bvh4_node* p, float lo[3][4], float hi[3][4], uint32_t c[4]) {
  const float4* q = reinterpret_cast<const float4*>(p);
  float4 v[7];
#pragma unroll
  for (int i = 0; i < 7; i++) v[i] = q[i];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    lo[a][0] = v[a].x, lo[a][1] = v[a].y, lo[a][2] = v[a].z, lo[a][3] = v[a].w;
    hi[a][0] = v[3 + a].x, hi[a][1] = v[3 + a].y, hi[a][2] = v[3 + a].z, hi[a][3] = v[3 + a].w;
  }
  c[0] = __float_as_uint(v[6].x), c[1] = __float_as_uint(v[6].y), c[2] = __float_as_uint(v[6].z), c[3] = __float_as_uint(v[6].w);
}

__device__ __forceinline__ void cswap(float t[4], uint32_t c[4], int i, int j) {
  if (t[j] < t[i]) {
    const float tt = t[i];
    t[i] = t[j], t[j] = tt;
    const uint32_t cc = c[i];
    c[i] = c[j], c[j] = cc;
  }
}

// Entry distances of the four slots of a node (+inf: missed or empty).
// All four slab tests run unconditionally and the empty slots are selected
// away afterwards, so the wave runs them as straight-line code.
__device__ __forceinline__ void node_slots(const tc_bvh4_node* node, const WoopRay& r, float tmin, float tmax, float t[4],
                                           uint32_t c[4]) {
  float lo[3][4], hi[3][4];
  load_node4(node, lo, hi, c);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const float bl[3] = {lo[0][k], lo[1][k], lo[2][k]}, bh[3] = {hi[0][k], hi[1][k], hi[2][k]};
    float bt = box_hit(r, bl, bh, tmin, tmax);
    asm volatile("" : "+v"(bt));  // keep the test out of a branch on the slot
    t[k] = c[k] == TC_BVH4_EMPTY ? INFINITY : bt;
  }
}

// (entry distance, child) of a slot as one double: the distance's bits are
// the high word, so doubles order as the distances do (negative ones, which
// only a negative tMin lets in, in reverse; the order of visits is a matter of
// speed alone), and one v_min_f64 / v_max_f64 pair swaps distance and child
// together.  A compare and four selects did that before.  The asm keeps
// fmin / fmax from quieting their operands first (the high words are never
// those of a NaN: an entry distance is a number or +inf).
__device__ __forceinline__ double slot_key(float t, uint32_t c) {
  return __longlong_as_double((long long)(((uint64_t)__float_as_uint(t) << 32) | c));
}
__device__ __forceinline__ void sort2(double& a, double& b) {
  double lo, hi;
  asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
  asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
  a = lo, b = hi;
}
__device__ __forceinline__ float key_t(double k) { return __uint_as_float((uint32_t)((uint64_t)__double_as_longlong(k) >> 32)); }
__device__ __forceinline__ uint32_t key_child(double k) { return (uint32_t)__double_as_longlong(k); }

// Where the near planes of a ray lie in a four-wide record: byte offsets of
// its lo or hi vector per axis, by the direction's sign; the far planes lie at
// the same offsets with the bits of kFarPlane flipped.
constexpr uint32_t kFarPlane[3] = {0x30, 0x50, 0x70};
__device__ __forceinline__ uint32_t near_plane(const WoopRay& r, int k) { return 16u * k + (r.inv[k] < 0.0f ? 48u : 0u); }

// Entry distances of the four slots of a node for regular rays: the planes
// are loaded in the order the ray meets them, so a slab takes no minimum and
// maximum (24 a node; the distances are the same bits), and an empty slot's
// inverted box (+inf, -inf) misses by itself.  `at` is the node's byte offset
// from the uniform `nodes`, below 4 GB, so the seven addresses are one register
// each.  A visit issues 130 vector instructions instead of 156; the trace
// launch takes 3832 -> 3727 us at patch field 3840 x 2160, 852 -> 835 us at 500
// meshes, 493 -> 481 us at grid64.
__device__ __forceinline__ void node_slots_ordered(const tc_bvh4_node* nodes, uint32_t at, const WoopRay& r,
                                                   const uint32_t near[3], float tmin, float tmax, float t[4], uint32_t c[4]) {
  const char* base = reinterpret_cast<const char*>(nodes);
  float4 n[3], f[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const uint32_t o = at | near[k];
    n[k] = gload(reinterpret_cast<const float4*>(base + o));
    f[k] = gload(reinterpret_cast<const float4*>(base + (o ^ kFarPlane[k])));
  }
  const uint4 ch = gload(reinterpret_cast<const uint4*>(base + (at | 96u)));
  c[0] = ch.x, c[1] = ch.y, c[2] = ch.z, c[3] = ch.w;
  const float nn[3][4] = {{n[0].x, n[0].y, n[0].z, n[0].w}, {n[1].x, n[1].y, n[1].z, n[1].w}, {n[2].x, n[2].y, n[2].z, n[2].w}};
  const float ff[3][4] = {{f[0].x, f[0].y, f[0].z, f[0].w}, {f[1].x, f[1].y, f[1].z, f[1].w}, {f[2].x, f[2].y, f[2].z, f[2].w}};
#pragma unroll
  for (int k = 0; k < 4; k++) {
    float tn = tmin, tf = tmax;
#pragma unroll
    for (int x = 0; x < 3; x++) {
      tn = fmaxf(tn, (nn[x][k] - r.o[x]) * r.inv[x]);
      tf = fminf(tf, (ff[x][k] - r.o[x]) * r.inv[x]);
    }
    float bt = tn <= tf * 1.0000005f ? tn : INFINITY;
    asm volatile("" : "+v"(bt));  // keep the test out of a branch on the slot
    t[k] = bt;
  }
}

// Visits one node: pushes the hit slots but the nearest (farthest first)
// and returns the nearest one's child, or pops when no slot is hit.  The top
// of the stack is read ahead of the box tests and every LDS entry is written
// whether its slot is hit or not; only the pointer advance depends on the
// hits (h hits move it by h - 1, one pop being -1), so the wave runs no branch.
// `ordered` is uniform: whether node_slots_ordered applies to every ray of the
// wave.
__device__ __forceinline__ uint32_t visit_node(const tc_bvh4_node* nodes, uint32_t first, uint32_t node, bool ordered,
                                               const WoopRay& r, const uint32_t near[3], float tmin, float tmax, RayStack& stack) {
  const uint32_t top = *stack.entry(min(stack.sp, kLdsStack * kStackStep) - kStackStep);
  float t[4];
  uint32_t c[4];
  if (ordered)
    node_slots_ordered(nodes, (first + node) * (uint32_t)sizeof(tc_bvh4_node), r, near, tmin, tmax, t, c);
  else
    node_slots(nodes + first + node, r, tmin, tmax, t, c);
  double k0 = slot_key(t[0], c[0]), k1 = slot_key(t[1], c[1]), k2 = slot_key(t[2], c[2]), k3 = slot_key(t[3], c[3]);
  sort2(k0, k1);
  sort2(k2, k3);
  sort2(k0, k2);
  sort2(k1, k3);
  sort2(k1, k2);
  const bool h0 = key_t(k0) != INFINITY, h1 = key_t(k1) != INFINITY, h2 = key_t(k2) != INFINITY, h3 = key_t(k3) != INFINITY;
  if (stack.sp + 2 * kStackStep < stack.ldsEnd) {
    uint32_t sp = stack.sp;
    *stack.entry(sp) = key_child(k3);
    sp += h3 ? kStackStep : 0u;
    *stack.entry(sp) = key_child(k2);
    sp += h2 ? kStackStep : 0u;
    *stack.entry(sp) = key_child(k1);
    sp += h1 ? kStackStep : 0u;
    stack.sp = h0 ? sp : sp - kStackStep;
    return h0 ? key_child(k0) : top;
  }
  if (!h0) return stack.pop();
  if (h3) stack.push(key_child(k3));
  if (h2) stack.push(key_child(k2));
  if (h1) stack.push(key_child(k1));
  return key_child(k0);
}

// LDS of one wave: the lanes' stacks and the state of a leaf step.
constexpr uint32_t kLeafQueue = 144;  // 15 left over + 128 of one step, rounded up
// Group pairs of a block, at most: its header counts 255 triangles
// (tc_cluster_template_order takes 256; clusters of the pipeline have 128 and
// 16 pairs).
constexpr uint32_t kBlockPairs = (255 + 2 * TC_CLAS_GROUP_TRIANGLES - 1) / (2 * TC_CLAS_GROUP_TRIANGLES);
struct WaveLds {
  uint32_t stack[kLdsStack * kWave];
  float4 rayO[kWave];          // origin, closest hit so far
  float4 rayI[kWave];          // inverse direction, tMin
  float4 rayS[kWave];          // shear, permutation | triangles << 8 | groups << 16
  uint4 leaf[kWave];           // CLAS address, (ordered t, primitive) of the closest hit
  float4 won[kWave];           // that hit's V, W, determinant and triangle word
  uint64_t heads[kBlockPairs]; // bit per group-box pair: the first of its lane
  uint32_t lanes[kWave];       // lanes with leaves, in order: lane | groups << 8 | first pair << 16
  uint16_t queue[kLeafQueue];  // groups entered: lane | group << 6
};

// Inclusive sum over the wave's lanes (all active).
__device__ __forceinline__ uint32_t wave_scan_dpp(uint32_t v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}

// Floats as unsigned words of the same order (-0 as 0).
__device__ __forceinline__ uint32_t ordered(float t) {
  const uint32_t u = __float_as_uint(t + 0.0f);
  return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}
__device__ __forceinline__ float from_ordered(uint32_t u) {
  return __uint_as_float((u & 0x80000000u) ? u ^ 0x80000000u : ~u);
}

// Closest hit of a ray; barycentrics are V / det and W / det.
struct BestHit {
  float t, V, W, det;
  uint32_t instanceID, clusterID, primitiveID;
  uint32_t word;     // triangle word
  const char* clas;  // CLAS block, null: no hit
};

__device__ __forceinline__ bool key_less(float t, uint32_t i, uint32_t c, uint32_t p, const BestHit& best) {
  if (t != best.t) return t < best.t;
  if (i != best.instanceID) return i < best.instanceID;
  if (c != best.clusterID) return c < best.clusterID;
  return p < best.primitiveID;
}

// Intersects the CLAS blocks that the wave's lanes hold (`has`), sharing the
// work over all 64 lanes; the whole wave calls it.  The traversal is bound by
// VALU issue (74 % busy at grid64), and what it issues is mostly idle lanes:
// about 22 of 64 lanes arrive with a leaf, their blocks hold 2 to 32 groups,
// and when each lane tested its own block's triangles 15 of 64 lanes were at
// work.  So every lane puts its ray in LDS, the group boxes of all blocks are
// numbered through (pairs of boxes, 48 bytes) and dealt one pair per lane,
// groups entered go to a queue, and the triangles of 16 queued groups at a
// time are dealt one per lane.  A candidate enters its ray's (t, primitive)
// minimum in LDS, so the result is that of testing one triangle after another.
// Measured against one lane per block (trace launch, same hits): grid64 552 ->
// 485 us, 500 meshes 1160 -> 856 us, patch field at 3840 x 2160 4975 -> 3850
// us, icosphere at 320 x 180 161 -> 132 us, parallel rays onto whole clusters
// (384^2 depth rays) 15.5 -> 17.5 us.
__device__ __forceinline__ void leaf_step(WaveLds& w, bool has, const char* clas, uint64_t info, const WoopRay& ray,
                                          float tmin, float tmax, bool cullBack, bool anyHit) {
  const uint32_t lane = lane_id();
  const uint32_t nt = (uint32_t)info & 0xFF, ng = ((uint32_t)info >> 16) & 0xFF;
  const uint32_t npairs = has ? min((ng + 1) >> 1, kBlockPairs) : 0;
  const uint32_t end = wave_scan_dpp(npairs), first = end - npairs;
  const uint32_t total = __builtin_amdgcn_readlane(end, 63);
  if (lane < kBlockPairs) w.heads[lane] = 0;
  wave_sync();
  // a block without triangles has no pairs: its first is its successor's, so it
  // takes no entry and no bit
  const uint64_t holders = ballot(npairs != 0);
  if (has) {
    const uint64_t addr = reinterpret_cast<uint64_t>(clas);
    w.rayO[lane] = make_float4(ray.o[0], ray.o[1], ray.o[2], tmax);
    w.rayI[lane] = make_float4(ray.inv[0], ray.inv[1], ray.inv[2], tmin);
    w.rayS[lane] = make_float4(ray.Sx, ray.Sy, ray.Sz,
                               __uint_as_float((uint32_t)(ray.kx | ray.ky << 2 | ray.kz << 4) | nt << 8 | ng << 16));
    w.leaf[lane] = make_uint4((uint32_t)addr, (uint32_t)(addr >> 32), ~0u, ~0u);
    if (npairs != 0) {
      w.lanes[mask_prefix(holders)] = lane | ng << 8 | first << 16;
      __hip_atomic_fetch_or(reinterpret_cast<uint32_t*>(w.heads) + (first >> 5), 1u << (first & 31), __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
  }
  wave_sync();
  // Which way the group boxes are tested, by what the two cost in units of
  // about 50 instructions: each lane its own block (one per pair of the largest
  // block, in steps of two pairs, and two to queue the groups) or the pairs
  // dealt out (two per 64 pairs).  Lanes that all hold whole clusters, as
  // under parallel rays, are better off with their own: 384^2 depth rays take
  // 17.5 us, 22.8 us with pairs always dealt out; steps of four pairs spill.
  uint32_t most = npairs;  // the wave's largest, in lane 63
  most = max(most, (uint32_t)__builtin_amdgcn_update_dpp(0, most, 0x111, 0xf, 0xf, true));
  most = max(most, (uint32_t)__builtin_amdgcn_update_dpp(0, most, 0x112, 0xf, 0xf, true));
  most = max(most, (uint32_t)__builtin_amdgcn_update_dpp(0, most, 0x114, 0xf, 0xf, true));
  most = max(most, (uint32_t)__builtin_amdgcn_update_dpp(0, most, 0x118, 0xf, 0xf, true));
  most = max(most, (uint32_t)__builtin_amdgcn_update_dpp(0, most, 0x142, 0xa, 0xf, false));
  most = max(most, (uint32_t)__builtin_amdgcn_update_dpp(0, most, 0x143, 0xc, 0xf, false));
  most = __builtin_amdgcn_readlane(most, 63);
  // (A lane's own groups are bits of one word.)
  const bool own = most <= 16 && (most == 1 ? 1 : (most + 1) & ~1u) + 2 <= 2 * ((total + kWave - 1) / kWave);
  uint32_t mask = 0;  // own: this lane's groups entered and not queued yet
  if (own) {
    const float4* gq = reinterpret_cast<const float4*>(clas + sizeof(tc_clas_header));
    mask = most == 1 ? group_mask<1>(ray, gq, npairs, tmin, tmax) : group_mask<2>(ray, gq, npairs, tmin, tmax);
    if (ng < 32) mask &= (1u << ng) - 1u;
  }
  uint32_t starts = 0, queued = 0;  // wave-uniform
  for (uint32_t base = 0;; base += kWave) {
    bool last;
    if (own) {
      const bool in = mask != 0;
      const uint64_t m = ballot(in);
      if (in) w.queue[queued + mask_prefix(m)] = (uint16_t)(lane | (uint32_t)__builtin_ctz(mask) << 6);
      mask &= mask - 1;
      queued += __popcll(m);
      last = !ballot(mask != 0);
    } else {
      last = base + kWave >= total;
      // the lane whose block holds pair base + lane: the number of first pairs
      // up to it
      const uint64_t heads = uniform64(w.heads[base / kWave]);
      const uint32_t at = starts + (uint32_t)(heads & 1) + mask_prefix(heads >> 1) - 1;
      starts += __popcll(heads);
      const bool valid = base + lane < total;
      bool in0 = false, in1 = false;
      uint32_t owner = 0, pair = 0;
      if (valid) {
        const uint32_t e = w.lanes[at];
        owner = e & 63;
        pair = base + lane - (e >> 16);
        const float4 ro = w.rayO[owner], ri = w.rayI[owner];
        const uint2 ca = *reinterpret_cast<const uint2*>(&w.leaf[owner]);
        const float4* gq =
            reinterpret_cast<const float4*>((((uint64_t)ca.y << 32) | ca.x) + sizeof(tc_clas_header) + pair * 48ull);
        const float4 a0 = gload(gq), a1 = gload(gq + 1), a2 = gload(gq + 2);
        WoopRay br;
        br.o[0] = ro.x, br.o[1] = ro.y, br.o[2] = ro.z;
        br.inv[0] = ri.x, br.inv[1] = ri.y, br.inv[2] = ri.z;
        in0 = group_hit(br, a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, ri.w, ro.w) != 0;
        in1 = 2 * pair + 1 < ((e >> 8) & 0xFF) && group_hit(br, a1.z, a1.w, a2.x, a2.y, a2.z, a2.w, ri.w, ro.w) != 0;
      }
      const uint64_t m0 = ballot(in0), m1 = ballot(in1);
      if (in0) w.queue[queued + mask_prefix(m0)] = (uint16_t)(owner | (2 * pair) << 6);
      queued += __popcll(m0);
      if (in1) w.queue[queued + mask_prefix(m1)] = (uint16_t)(owner | (2 * pair + 1) << 6);
      queued += __popcll(m1);
    }
    wave_sync();
    // triangles of the queued groups, 16 groups at a time (all that is left
    // after the last pairs)
    uint32_t q = 0;
    for (; q + 16 <= queued || (last && q < queued); q += 16) {
      const uint32_t k = q + (lane >> 2);
      uint32_t who = 0;
      uint64_t key = ~0ull;
      float V = 0.f, W = 0.f, det = 1.f;
      uint32_t word = 0;
      bool hit = false;
      if (k < queued) {
        const uint32_t e = w.queue[k];
        who = e & 63;
        const uint32_t tri = (e >> 6) * TC_CLAS_GROUP_TRIANGLES + (lane & 3);
        const float4 rs = w.rayS[who];
        const uint32_t code = __float_as_uint(rs.w);
        const uint32_t bnt = (code >> 8) & 0xFF, bng = code >> 16;
        if (tri < bnt) {
          const uint2 ca = *reinterpret_cast<const uint2*>(&w.leaf[who]);
          const char* tris = reinterpret_cast<const char*>(((uint64_t)ca.y << 32) | ca.x) + sizeof(tc_clas_header) +
                             ((bng * 24u + 15u) & ~15u);
          word = gload(reinterpret_cast<const uint32_t*>(tris) + tri);
          const float* verts = reinterpret_cast<const float*>(tris + ((bnt * 4u + 15u) & ~15u));
          const gfloat3 p0 = gld3(verts + 3 * (word & 0xFF)), p1 = gld3(verts + 3 * ((word >> 8) & 0xFF)),
                        p2 = gld3(verts + 3 * ((word >> 16) & 0xFF));
          const float4 ro = w.rayO[who];
          WoopRay tr;
          tr.o[0] = ro.x, tr.o[1] = ro.y, tr.o[2] = ro.z;
          tr.kx = code & 3, tr.ky = (code >> 2) & 3, tr.kz = (code >> 4) & 3;
          tr.Sx = rs.x, tr.Sy = rs.y, tr.Sz = rs.z;
          const float q0[3] = {p0.x, p0.y, p0.z}, q1[3] = {p1.x, p1.y, p1.z}, q2[3] = {p2.x, p2.y, p2.z};
          TriDet h;
          if (tri_test(tr, q0, q1, q2, cullBack, w.rayI[who].w, ro.w, h)) {
            hit = true;
            key = ((uint64_t)ordered(h.t) << 32) | (word >> 24);
            V = h.V, W = h.W, det = h.det;
          }
        }
      }
      uint64_t* best = reinterpret_cast<uint64_t*>(&w.leaf[who].z);
      if (hit) {
        if (anyHit)
          *best = 0;
        else
          __hip_atomic_fetch_min(best, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      }
      wave_sync();
      if (hit && !anyHit && *best == key) w.won[who] = make_float4(V, W, det, __uint_as_float(word));
      wave_sync();
    }
    if (last) break;
    // the groups left over move to the front
    const uint32_t left = queued - q;
    uint32_t e = 0;
    if (lane < left) e = w.queue[q + lane];
    wave_sync();
    if (lane < left) w.queue[lane] = (uint16_t)e;
    queued = left;
    wave_sync();
  }
}

// Full two-level traversal of the wave's rays (the lanes with `live`) over
// the four-wide views; the whole wave calls it.  Returns true in the lanes
// whose ray hit anything.  The TLAS walk stops at each instance whose BLAS
// has clusters; that BLAS is walked with the object-space ray until its stack
// sentinel is popped.
__device__ __forceinline__ bool trace_wave(const TraceArgs& a, WaveLds& w, RayStack& stack, const float o[3], const float d[3],
                                           float tmin, float tmax, bool live, bool cullBack, bool anyHit, BestHit& best) {
  best.t = tmax;
  best.V = best.W = 0.0f;
  best.det = 1.0f;
  best.instanceID = best.clusterID = best.primitiveID = 0xFFFFFFFFu;
  best.word = 0;
  best.clas = nullptr;
  bool found = false;
  WoopRay world;
  setup_box_ray(world, o, d);
  uint32_t worldNear[3];
  for (int k = 0; k < 3; k++) worldNear[k] = near_plane(world, k);
  // (a plane through the origin of a ray parallel to it gives 0 * inf, which
  // the general test reads as a miss)
  const bool worldOrdered = a.nodes32 && !ballot(live && !regular_ray(world));
  stack.sp = 0;
  stack.push(kDone);
  uint32_t e = live ? *a.tlasRoot : kDone;
  while (true) {
    // TLAS: find the next instance leaf with clusters
    uint32_t inst = kDone;
    while (e != kDone) {
      if (e & TC_BVH_LEAF) {
        const uint32_t i = e & 0x3FFFFFFFu;
        if (a.tlasInstances[i].numClusters != 0) {
          inst = i;
          break;
        }
        e = stack.pop();
      } else {
        e = visit_node(a.tlasNodes4, 0, e, worldOrdered, world, worldNear, tmin, best.t, stack);
      }
    }
    if (!ballot(inst != kDone)) break;
    WoopRay ray;
    uint32_t first = 0, near[3] = {0, 0, 0};  // the instance's first node
    bool irregular = false;
    const uint64_t* leafAddr = nullptr;
    const uint64_t* leafInfo = nullptr;
    uint32_t b = kDone;
    if (inst != kDone) {
      const tc_tlas_instance& ti = a.tlasInstances[inst];
      float ol[3], dl[3];
      xform34(ti.worldToObject, o, 1.0f, ol);
      xform34(ti.worldToObject, d, 0.0f, dl);
      setup_ray(ray, ol, dl);
      for (int k = 0; k < 3; k++) near[k] = near_plane(ray, k);
      irregular = !regular_ray(ray);
      first = (uint32_t)((ti.blasNodes - a.blasNodesBase) / sizeof(tc_bvh_node));
      leafAddr = reinterpret_cast<const uint64_t*>(ti.blasLeaves);
      leafInfo = a.blasLeafInfo + (ti.blasLeaves - a.blasLeavesBase) / 8;
      stack.push(kDone);
      b = ti.blasRoot;
    }
    const bool ordered = a.nodes32 && !ballot(irregular);
    while (true) {
      // lanes walk nodes until each holds a CLAS leaf or has finished, or too
      // few still search
      while (true) {
        const uint64_t searching = ballot((int32_t)b >= 0);
        if (!searching) break;
        if ((uint32_t)__popcll(searching) * kSearchShare < (uint32_t)__popcll(ballot(b != kDone))) break;
        if ((int32_t)b >= 0) b = visit_node(a.blasNodes4, first, b, ordered, ray, near, tmin, best.t, stack);
      }
      const bool has = (int32_t)b < 0 && b != kDone;
      if (!ballot(has)) break;
      const char* clas = nullptr;
      uint64_t info = 0;
      if (has) {
        clas = reinterpret_cast<const char*>(gload(leafAddr + (b & ~TC_BVH_LEAF)));
        info = gload(leafInfo + (b & ~TC_BVH_LEAF));
      }
      leaf_step(w, has, clas, info, ray, tmin, best.t, cullBack, anyHit);
      if (has) {
        const uint32_t lane = lane_id();
        const uint4 lf = w.leaf[lane];
        const uint32_t clusterID = (uint32_t)(info >> 32);
        if ((lf.z & lf.w) != ~0u) {
          const float t = from_ordered(lf.w);
          if (anyHit) {
            found = true;
          } else if (key_less(t, inst, clusterID, lf.z, best)) {
            const float4 won = w.won[lane];
            best.t = t;
            best.V = won.x, best.W = won.y, best.det = won.z;
            best.word = __float_as_uint(won.w);
            best.instanceID = inst, best.clusterID = clusterID, best.primitiveID = lf.z;
            best.clas = clas;
          }
        }
        b = found ? kDone : stack.pop();
      }
      wave_sync();
    }
    if (inst != kDone) e = found ? kDone : stack.pop();
  }
  return anyHit ? found : best.instanceID != 0xFFFFFFFFu;
}

// Wave-wide packet traversal: the 64 lanes of a wave walk one shared node
// stack (in LDS, uniform entries).  A node is entered when any live lane's
// ray enters it before that lane's current closest hit, so every lane sees
// a superset of the nodes its own traversal would visit and finds the same
// closest hit (ties are broken by key).  Node records are fetched once per
// wave.  Suited to coherent rays: camera rays in 8 x 8 pixel tiles and their
// shadow rays.
constexpr uint32_t kPacketStack = 160;
static_assert(kMostEntries <= kPacketStack, "entries of the deepest trees");
constexpr uint32_t kBlasEntry = 1u << 30;  // packet stack: marks BLAS entries

__device__ __forceinline__ float wave_min_f(float v) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) v = fminf(v, __shfl_xor(v, d, kWave));
  return v;
}

__device__ bool trace_packet(const TraceArgs& a, const float o[3], const float d[3], float tmin, float tmax, bool live,
                             bool cullBack, bool anyHit, uint32_t* stk, HitState& best) {
  best.h.t = tmax;
  best.h.u = best.h.v = 0.0f;
  best.h.instanceID = best.h.clusterID = best.h.primitiveID = 0xFFFFFFFFu;
  best.clas = nullptr;
  best.word = 0;
  WoopRay world, ray;
  setup_ray(world, o, d);
  ray = world;
  uint32_t sp = 0;
  uint32_t e = __builtin_amdgcn_readfirstlane(*a.tlasRoot);
  uint32_t inst = 0xFFFFFFFFu;
  const tc_bvh4_node* blas4 = nullptr;
  const uint64_t* blasLeaves = nullptr;
  const uint64_t* leafInfo = nullptr;
  bool found = false;
  while (true) {
    if (!ballot(live)) break;
    bool next = false;  // pop the next entry
    if (!(e & kBlasEntry)) {
      if (inst != 0xFFFFFFFFu) {
        ray = world;
        inst = 0xFFFFFFFFu;
      }
      if (e & TC_BVH_LEAF) {
        const uint32_t i = e & 0x3FFFFFFFu;
        const tc_tlas_instance& ti = a.tlasInstances[i];
        if (ti.numClusters != 0) {
          float ol[3], dl[3];
          xform34(ti.worldToObject, o, 1.0f, ol);
          xform34(ti.worldToObject, d, 0.0f, dl);
          setup_ray(ray, ol, dl);
          inst = i;
          blas4 = a.blasNodes4 + (ti.blasNodes - a.blasNodesBase) / sizeof(tc_bvh_node);
          blasLeaves = reinterpret_cast<const uint64_t*>(ti.blasLeaves);
          leafInfo = a.blasLeafInfo + (ti.blasLeaves - a.blasLeavesBase) / 8;
          e = __builtin_amdgcn_readfirstlane(kBlasEntry | ti.blasRoot);
          continue;
        }
        next = true;
      }
    } else if (e & TC_BVH_LEAF) {
      const uint32_t leaf = e & ~(kBlasEntry | TC_BVH_LEAF);
      const char* clas = reinterpret_cast<const char*>(blasLeaves[leaf]);
      if (live && clas_hit(ray, clas, leafInfo[leaf], inst, cullBack, anyHit, tmin, best)) {
        found = true;
        live = false;  // any-hit: this lane is done
      }
      next = true;
    }
    if (!next) {
      const tc_bvh4_node* node = (e & kBlasEntry) ? blas4 + (e & ~kBlasEntry) : a.tlasNodes4 + e;
      const uint32_t tag = e & kBlasEntry;
      float lo[3][4], hi[3][4], t[4], tw[4];
      uint32_t c[4];
      load_node4(node, lo, hi, c);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const float bl[3] = {lo[0][k], lo[1][k], lo[2][k]}, bh[3] = {hi[0][k], hi[1][k], hi[2][k]};
        float bt = box_hit(ray, bl, bh, tmin, best.h.t);
        asm volatile("" : "+v"(bt));
        t[k] = (c[k] == TC_BVH4_EMPTY || !live) ? INFINITY : bt;
        tw[k] = wave_min_f(t[k]);  // nearest entry over the packet (uniform)
        c[k] |= tag;
      }
      cswap(tw, c, 0, 1);
      cswap(tw, c, 2, 3);
      cswap(tw, c, 0, 2);
      cswap(tw, c, 1, 3);
      cswap(tw, c, 1, 2);
      if (tw[0] == INFINITY) {
        next = true;
      } else {
        if (tw[3] != INFINITY && sp < kPacketStack) stk[sp++] = c[3];
        if (tw[2] != INFINITY && sp < kPacketStack) stk[sp++] = c[2];
        if (tw[1] != INFINITY && sp < kPacketStack) stk[sp++] = c[1];
        e = __builtin_amdgcn_readfirstlane(c[0]);
      }
    }
    if (next) {
      if (sp == 0) break;
      e = __builtin_amdgcn_readfirstlane(stk[--sp]);
    }
  }
  return anyHit ? found : best.h.instanceID != 0xFFFFFFFFu;
}

__device__ __forceinline__ void mul44(const float* m, const float v[4], float out[4]) {
#pragma unroll
  for (int r = 0; r < 4; r++) out[r] = ((m[r] * v[0] + m[4 + r] * v[1]) + m[8 + r] * v[2]) + m[12 + r] * v[3];
}

__device__ __forceinline__ void normalize4(float v[4]) {
  const float l = sqrtf(((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]) + v[3] * v[3]);
  const float s = 1.0f / l;
  for (int k = 0; k < 4; k++) v[k] = v[k] * s;
}

// Camera rays come in 8 x 8 pixel tiles, one per wave.  Consecutive
// workgroups go to the eight XCDs in turn, so wave w of a launch runs on XCD
// (w / wavesPerGroup) % 8.  The image is cut into eight vertical strips of
// tiles and the waves of XCD x walk strip x in row order, so each XCD's L2
// holds the geometry seen through one strip.  Strips differ in width by at
// most one tile; a wave past the end of its strip has no tile (false).  With
// `rowOrder` the strip's rows are walked in that order instead (a
// permutation of the tile rows, TraceOrder).
constexpr uint32_t kXcds = 8;

// A wave's tile time into its row's maximum (no return value: the wave does
// not wait for it).
__device__ __forceinline__ void time_tile_row(TraceOrder* ord, uint32_t row, uint64_t t0) {
  const uint64_t dt = __builtin_amdgcn_s_memrealtime() - t0;
  __hip_atomic_fetch_max(&ord->rowTime[row], (uint32_t)min(dt, (uint64_t)0xFFFFFFFFu), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
}

__host__ __device__ __forceinline__ uint32_t strip_waves(uint32_t tilesX, uint32_t tilesY, uint32_t wavesPerGroup) {
  const uint32_t perXcd = (tilesX + kXcds - 1) / kXcds * tilesY;
  return kXcds * ((perXcd + wavesPerGroup - 1) / wavesPerGroup) * wavesPerGroup;
}

__device__ __forceinline__ bool strip_tile(uint32_t w, uint32_t wavesPerGroup, uint32_t tilesX, uint32_t tilesY,
                                           const uint32_t* rowOrder, uint32_t& tx, uint32_t& ty) {
  const uint32_t b = w / wavesPerGroup, x = b % kXcds;
  const uint32_t k = (b / kXcds) * wavesPerGroup + w % wavesPerGroup;
  const uint32_t c0 = x * tilesX / kXcds, sw = (x + 1) * tilesX / kXcds - c0;
  if (sw == 0 || k / sw >= tilesY) return false;
  tx = c0 + k % sw;
  ty = rowOrder ? rowOrder[uniform(k / sw)] : k / sw;
  return true;
}


// render_raytrace.rgen.glsl:52-86
__device__ __forceinline__ void primary_ray(const tc_frame_constants* view, uint32_t x, uint32_t y, uint32_t W, uint32_t H,
                                            float o[3], float d[3]) {
  const float uvx = ((float)x + 0.5f) / (float)W, uvy = ((float)y + 0.5f) / (float)H;
  const float dx = uvx * 2.0f - 1.0f, dy = uvy * 2.0f - 1.0f;
  const float org[4] = {0.0f, 0.0f, 0.0f, 1.0f};
  float origin[4];
  mul44(view->viewMatrixI, org, origin);
  const float ndc[4] = {dx, dy, 1.0f, 1.0f};
  float target[4];
  mul44(view->projMatrixI, ndc, target);
  normalize4(target);
  const float tv[4] = {target[0], target[1], target[2], 0.0f};
  float dir[4];
  mul44(view->viewMatrixI, tv, dir);
  normalize4(dir);
  for (int k = 0; k < 3; k++) o[k] = origin[k], d[k] = dir[k];
}

// render_raytrace_clusters.rchit.glsl:128-236 and 338-339: base cluster,
// triangle and barycentrics, world position and depth of a hit
__device__ void decode_hit(const TraceArgs& a, const HitState& hs, tc_hit_decoded& out) {
  const tc_hit& h = hs.h;
  out.instanceID = h.instanceID;
  out.shadowed = 0;
  if (h.instanceID == 0xFFFFFFFFu) {
    out.clusterID = out.triangleID = out.subTriangleID = 0xFFFFFFFFu;
    out.baryBase[0] = out.baryBase[1] = out.baryBase[2] = 0.0f;
    out.depth = 1.0f;
    out.wPos[0] = out.wPos[1] = out.wPos[2] = 0.0f;
    return;
  }
  const uint32_t mode = h.clusterID >> 30;
  uint32_t clusterID = h.clusterID & 0x3FFFFFFFu;
  uint32_t triangleID = h.primitiveID;
  uint32_t subTriangle = h.primitiveID;
  const v3 bw = mk((1.0f - h.u) - h.v, h.u, h.v);
  v3 base = bw;
  if (mode == TC_RT_CLUSTER_MODE_1X_SUBSET_CLUSTER) {
    // :173-178 the part slot holds the ClusterInfo, then one byte per
    // transient triangle naming the cluster triangle
    const uint8_t* slot = ptr<const uint8_t>(a.build->partTriangles) + (uint64_t)clusterID * 24ull;
    const tc_cluster_info ci = *reinterpret_cast<const tc_cluster_info*>(slot);
    triangleID = slot[8 + h.primitiveID];
    clusterID = ci.clusterID;
  } else if (mode == TC_RT_CLUSTER_MODE_2X_BATCHED_TESSELLATED) {
    // :152-170 a u16 mapping per batch triangle after the ClusterInfo: the
    // cluster triangle, the sub-triangle of its config (masked with 0xF; the
    // reference's `& 4` drops sub-triangles 1-3) and the (factor - 1) bits
    // the config is rebuilt from
    const uint8_t* slot = ptr<const uint8_t>(a.build->partTriangles) + (uint64_t)clusterID * 24ull;
    const tc_cluster_info ci = *reinterpret_cast<const tc_cluster_info*>(slot);
    const uint32_t packed = reinterpret_cast<const uint16_t*>(slot + 8)[h.primitiveID];
    triangleID = packed & 0xFFu;
    subTriangle = (packed >> 8) & 0xFu;
    uint32_t f[3] = {1u + ((packed >> 12) & 1u), 1u + ((packed >> 13) & 1u), 1u + (packed >> 14)};
    uint32_t vtx[3] = {0u, 32768u, 32768u << 16};
    const uint32_t cfg = get_config(f, vtx);
    clusterID = ci.clusterID;
    const TableView T = load_table(a.tessTable);
    const tc_tess_table_entry e = cfg_entry(T, cfg);
    uint32_t idx[3];
    cfg_tri_vertices(T, cfg, e.firstTriangle, subTriangle, idx);
    const v3 nb = interp(cfg_vertex_bary(T, cfg, e.firstVertex, idx[0]), cfg_vertex_bary(T, cfg, e.firstVertex, idx[1]),
                         cfg_vertex_bary(T, cfg, e.firstVertex, idx[2]), bw);
    base = interp(decode_bary(vtx[0]), decode_bary(vtx[1]), decode_bary(vtx[2]), nb);
  } else if (mode != TC_RT_CLUSTER_MODE_FULL_CLUSTER) {
    const tc_tess_triangle_info ti = ptr<const tc_tess_triangle_info>(a.build->partTriangles)[clusterID];
    triangleID = ti.subTriangle.triangleID_config & 0xFFFF;
    const uint32_t cfg = ti.subTriangle.triangleID_config >> 16;
    clusterID = ti.cluster.clusterID;
    const TableView T = load_table(a.tessTable);
    const tc_tess_table_entry e = cfg_entry(T, cfg);
    uint32_t idx[3];
    cfg_tri_vertices(T, cfg, e.firstTriangle, h.primitiveID, idx);
    const v3 nb = interp(cfg_vertex_bary(T, cfg, e.firstVertex, idx[0]), cfg_vertex_bary(T, cfg, e.firstVertex, idx[1]),
                         cfg_vertex_bary(T, cfg, e.firstVertex, idx[2]), bw);
    base = interp(decode_bary(ti.subTriangle.vtxEncoded[0]), decode_bary(ti.subTriangle.vtxEncoded[1]),
                  decode_bary(ti.subTriangle.vtxEncoded[2]), nb);
  }
  out.clusterID = clusterID;
  out.triangleID = triangleID;
  out.subTriangleID = subTriangle;
  out.baryBase[0] = base.x, out.baryBase[1] = base.y, out.baryBase[2] = base.z;
  // :248-249 object-space hit point from the hit triangle, then world
  const tc_clas_header hdr = *reinterpret_cast<const tc_clas_header*>(hs.clas);
  const float* verts = clas_vertices(hs.clas, hdr.counts & 0xFF, (hdr.counts >> 16) & 0xFF);
  const float* p0 = verts + 3 * (hs.word & 0xFF);
  const float* p1 = verts + 3 * ((hs.word >> 8) & 0xFF);
  const float* p2 = verts + 3 * ((hs.word >> 16) & 0xFF);
  const v3 op = interp(mk(p0[0], p0[1], p0[2]), mk(p1[0], p1[1], p1[2]), mk(p2[0], p2[1], p2[2]), bw);
  const float opv[3] = {op.x, op.y, op.z};
  float wp[3];
  xform34(a.tlasInstances[h.instanceID].objectToWorld, opv, 1.0f, wp);
  out.wPos[0] = wp[0], out.wPos[1] = wp[1], out.wPos[2] = wp[2];
  const float w4[4] = {wp[0], wp[1], wp[2], 1.0f};
  float pp[4];
  mul44(a.view->viewProjMatrix, w4, pp);
  out.depth = pp[2] / pp[3];
}

// Waves a tile's (or 64 explicit rays') rays are dealt over, as a power of two.
// A launch that leaves most of the chip's waves empty takes as long as its
// longest wave, which visits the nodes of all its rays: with fewer rays a wave
// that chain is shorter, and the leaf steps use the idle lanes all the same.
// While the shared waves are resident together (16 a CU; 6 for explicit rays,
// which also come in parallel bundles that want whole waves), down to four
// rays a wave: 160 x 90 / 320 x 180 camera rays onto 500 meshes 600 -> 244, 595 ->
// 349 us, onto an icosphere 124 -> 92, 132 -> 98.  The first halving up to 24 a
// CU: 480 x 270 / 560 x 315 500 meshes 562 -> 462, 548 -> 430, icosphere 138 -> 119,
// 129 -> 121, 64 grids 207 -> 169, 222 -> 191; past it 640 x 360 150 -> 156 and
// 960 x 540 191 -> 227.  (The further halvings up to 24 a CU, at 256 x 144: 500
// meshes 359 -> 279, but icosphere 94 -> 102 and 25 meshes 108 -> 121.)  16384
// vertical rays onto whole clusters 12.4 -> 10.2 us and onto parts 26 -> 18, 65536
// of them 13.6 -> 14.9 and 28 -> 25.
constexpr uint32_t kMaxShare = 4;
static uint32_t tile_share(uint32_t waves, bool rays) {
  const uint64_t cus = num_cu_public();
  uint32_t s = 0;
  while (s < kMaxShare && ((uint64_t)waves << (s + 1)) <= cus * (rays ? 6u : s == 0 ? 24u : 16u)) s++;
  return s;
}

// One ray per lane, up to 64 rays per wave.  The primary and the shadow walk are
// two rounds of one loop, so the traversal is one piece of code in the
// instruction cache.  A wave's lanes stay together through both: lanes without
// a ray (ragged tiles, rays past the end, misses in the shadow round) help in
// the leaf steps.
template <uint32_t T>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_trace(TraceArgs a) {
  __shared__ WaveLds s_wave[T / kWave];
  uint32_t spill[kStackDepth];
  WaveLds& w = s_wave[threadIdx.x / kWave];
  const uint32_t lane = lane_id();
  RayStack stack;
  stack.lds = (lds_u32*)(w.stack + lane);
  stack.spill = (private_u32*)spill;
  stack.ldsEnd = (a.flags & TC_TRACE_PRIVATE_STACK) ? 0u : kLdsStack * kStackStep;
  stack.sp = 0;
  const bool cull = (a.flags & TC_TRACE_CULL_BACK) != 0;
  const bool shadows = (a.flags & TC_TRACE_SHADOW) != 0 && a.decoded;
  const uint32_t tilesX = (a.width + 7) / 8, tilesY = (a.height + 7) / 8;
  // tile-row order: the last ranking when it ranked this many rows.  Each
  // wave's tile time goes to its row by an atomic nobody waits for.
  TraceOrder* ord = !a.rays && a.order && tilesY <= kMaxOrderRows ? a.order : nullptr;
  const uint32_t* rowOrder = ord && ord->rows == tilesY ? ord->order : nullptr;
  if (ord && blockIdx.x == 0 && threadIdx.x == 0) ord->pendingRows = tilesY;
  const uint32_t waves = gridDim.x * (T / kWave), perWave = kWave >> a.share, numWaves = (a.numItems + perWave - 1) / perWave;
  for (uint32_t wave = uniform(blockIdx.x * (T / kWave) + threadIdx.x / kWave); wave < numWaves; wave += waves) {
    const uint64_t t0 = ord ? __builtin_amdgcn_s_memrealtime() : 0;
    float o[3] = {0.f, 0.f, 0.f}, d[3] = {0.f, 0.f, 1.f}, tmin = 0.f, tmax = 0.f;
    bool live = false;
    uint32_t r = 0, timedRow = 0;
    if (a.rays) {
      r = wave * perWave + lane;
      live = lane < perWave && r < a.numItems;
      if (live) {
        const tc_ray ray = a.rays[r];
        for (int k = 0; k < 3; k++) o[k] = ray.origin[k], d[k] = ray.direction[k];
        tmin = ray.tMin;
        tmax = ray.tMax;
      }
    } else {
      uint32_t tx, ty;
      // the waves that share a tile are eight workgroups apart, on one XCD
      const uint32_t group = wave / (T / kWave), turn = group / kXcds, part = turn & ((1u << a.share) - 1u);
      const uint32_t tile = ((turn >> a.share) * kXcds + group % kXcds) * (T / kWave) + wave % (T / kWave);
      if (!strip_tile(tile, T / kWave, tilesX, tilesY, rowOrder, tx, ty)) continue;
      timedRow = ty;
      const uint32_t in = part * perWave + lane, x = tx * 8 + (in & 7), y = ty * 8 + (in >> 3);
      live = lane < perWave && x < a.width && y < a.height;
      if (live) {
        r = y * a.width + x;
        primary_ray(a.view, x, y, a.width, a.height, o, d);
        tmin = a.view->nearPlane;
        tmax = a.view->farPlane;
      }
    }
#pragma nounroll
    for (uint32_t round = 0; round < 2; round++) {
      BestHit best;
      const bool any = trace_wave(a, w, stack, o, d, tmin, tmax, live, cull && round == 0, round != 0, best);
      if (round != 0) {
        // render_shading.glsl:263-274: opaque, terminated on the first hit
        if (live && any) a.decoded[r].shadowed = 1u;
        break;
      }
      HitState hs;
      hs.h.t = any ? best.t : -1.0f;
      hs.h.u = best.V / best.det, hs.h.v = best.W / best.det;
      hs.h.instanceID = best.instanceID, hs.h.clusterID = best.clusterID, hs.h.primitiveID = best.primitiveID;
      hs.clas = best.clas, hs.word = best.word;
      bool shade = false;
      if (live) {
        if (a.hits) a.hits[r] = hs.h;
        if (a.hitVertices) {
          uint4 hv = make_uint4(~0u, ~0u, ~0u, ~0u);
          if (hs.clas) {
            const uint32_t base = reinterpret_cast<const tc_clas_header*>(hs.clas)->vertexBase;
            hv = make_uint4(base + (hs.word & 0xFF), base + ((hs.word >> 8) & 0xFF), base + ((hs.word >> 16) & 0xFF), 0u);
          }
          reinterpret_cast<uint4*>(a.hitVertices)[r] = hv;
        }
        if (a.decoded) {
          tc_hit_decoded dec;
          decode_hit(a, hs, dec);
          a.decoded[r] = dec;
          shade = shadows && any;
          for (int k = 0; k < 3; k++) o[k] = dec.wPos[k];
        }
      }
      if (!ballot(shade)) break;
      // the shadow ray of every hit
      live = shade;
      for (int k = 0; k < 3; k++) d[k] = a.view->skyParams.sunDirection[k];
      tmin = 0.001f;
      tmax = 10000000.0f;
    }
    if (ord && lane == 0) time_tile_row(ord, timedRow, t0);
  }
}

// Packet form of k_trace: one wave per 64 work items (an 8 x 8 pixel tile
// for camera rays), shared stack per wave.
template <uint32_t T>
__global__ __launch_bounds__(T) void k_trace_packet(TraceArgs a) {
  __shared__ uint32_t s_stk[T / kWave][kPacketStack];
  const uint32_t wave = threadIdx.x / kWave, lane = lane_id();
  uint32_t* stk = s_stk[wave];
  const bool cull = (a.flags & TC_TRACE_CULL_BACK) != 0;
  const bool shadows = (a.flags & TC_TRACE_SHADOW) != 0 && a.decoded;
  const uint32_t tilesX = (a.width + 7) / 8, tilesY = (a.height + 7) / 8;
  const uint32_t wavesTotal = gridDim.x * (T / kWave);
  for (uint32_t base = (blockIdx.x * (T / kWave) + wave) * kWave; base < a.numItems; base += wavesTotal * kWave) {
    const uint32_t item = base + lane;
    float o[3] = {0.f, 0.f, 0.f}, d[3] = {0.f, 0.f, 1.f}, tmin = 0.f, tmax = 0.f;
    uint32_t r = 0xFFFFFFFFu;
    if (item < a.numItems) {
      if (a.rays) {
        r = item;
        const tc_ray ray = a.rays[r];
        for (int k = 0; k < 3; k++) o[k] = ray.origin[k], d[k] = ray.direction[k];
        tmin = ray.tMin;
        tmax = ray.tMax;
      } else {
        uint32_t tx = 0, ty = 0;
        const bool tiled = strip_tile(item >> 6, T / kWave, tilesX, tilesY, nullptr, tx, ty);
        const uint32_t in = item & 63, x = tx * 8 + (in & 7), y = ty * 8 + (in >> 3);
        if (tiled && x < a.width && y < a.height) {
          r = y * a.width + x;
          primary_ray(a.view, x, y, a.width, a.height, o, d);
          tmin = a.view->nearPlane;
          tmax = a.view->farPlane;
        }
      }
    }
    const bool live = r != 0xFFFFFFFFu;
    HitState hs;
    trace_packet(a, o, d, tmin, tmax, live, cull, false, stk, hs);
    tc_hit hit = hs.h;
    if (hit.instanceID == 0xFFFFFFFFu) hit.t = -1.0f;
    tc_hit_decoded dec;
    if (live) {
      if (a.hits) a.hits[r] = hit;
      if (a.hitVertices) {
        uint4 hv = make_uint4(~0u, ~0u, ~0u, ~0u);
        if (hs.clas) {
          const uint32_t vb = reinterpret_cast<const tc_clas_header*>(hs.clas)->vertexBase;
          hv = make_uint4(vb + (hs.word & 0xFF), vb + ((hs.word >> 8) & 0xFF), vb + ((hs.word >> 16) & 0xFF), 0u);
        }
        reinterpret_cast<uint4*>(a.hitVertices)[r] = hv;
      }
      if (a.decoded) decode_hit(a, hs, dec);
    }
    if (shadows) {
      // render_shading.glsl:263-274: opaque, terminate on first hit
      const bool sLive = live && hit.instanceID != 0xFFFFFFFFu;
      const float* sun = a.view->skyParams.sunDirection;
      const float sd[3] = {sun[0], sun[1], sun[2]};
      const float so[3] = {sLive ? dec.wPos[0] : 0.f, sLive ? dec.wPos[1] : 0.f, sLive ? dec.wPos[2] : 0.f};
      HitState sh;
      const bool shadowed = trace_packet(a, so, sd, 0.001f, 10000000.0f, sLive, false, true, stk, sh);
      if (sLive) dec.shadowed = shadowed ? 1u : 0u;
    }
    if (live && a.decoded) a.decoded[r] = dec;
  }
}

}  // namespace tc

using namespace tc;

tc_status tc::trace_rays(const tc_bindings* b, tc_config config, const tc_accel* accel, const tc_trace_params* p,
                         TraceOrder* order, tc_stream stream) {
  KArgs ka;
  tc_status s = make_args_public(b, config, ka);
  if (s != TC_OK) return s;
  if (!accel || !p || !accel->tlasInstances || !accel->blasLeafInfo || (!p->hits && !p->decoded && !p->hitVertices))
    return TC_ERROR_INVALID_ARGUMENT;
  TraceArgs a;
  a.view = b->view;
  a.tessTable = b->tessTable;
  a.build = b->build;
  a.tlasInstances = accel->tlasInstances;
  a.tlasNodes = accel->tlasNodes;
  a.tlasRoot = accel->tlasRoot;
  a.rays = p->rays;
  a.width = p->width;
  a.height = p->height;
  a.numRays = p->rays ? p->numRays : p->width * p->height;
  a.tlasNodes4 = accel->tlasNodes4;
  a.blasNodes4 = accel->blasNodes4;
  a.blasNodesBase = reinterpret_cast<uint64_t>(accel->blasNodes);
  a.blasLeavesBase = reinterpret_cast<uint64_t>(accel->blasLeaves);
  a.blasLeafInfo = accel->blasLeafInfo;
  a.hits = p->hits;
  a.decoded = p->decoded;
  a.hitVertices = p->hitVertices;
  a.order = order;
  // byte offsets of every node fit 32 bits
  a.nodes32 = (uint64_t)std::max(accel->capacity, accel->numInstances) * sizeof(tc_bvh4_node) <= 0xFFFFFFFFull;
  a.flags = p->flags;
  if (!p->rays && (!p->width || !p->height)) return TC_ERROR_INVALID_ARGUMENT;
  if (a.numRays == 0) return TC_OK;
  const tc_tuning tn = tuning_snapshot();
  const uint32_t T = tn.traceThreads;
  a.numItems = p->rays ? p->numRays : strip_waves((p->width + 7) / 8, (p->height + 7) / 8, T / kWave) * kWave;
  a.share = (a.flags & TC_TRACE_PACKETS) ? 0u : tile_share((a.numItems + kWave - 1) / kWave, p->rays != nullptr);
  const uint32_t grid = std::min<uint32_t>((((uint64_t)a.numItems << a.share) + T - 1) / T, (uint32_t)num_cu_public() * tn.traceBlocksPerCU);
  // resident waves: four per SIMD (128 VGPRs), four SIMDs per CU
  if ((uint64_t)grid * (T / kWave) > (uint64_t)kOrderRounds * num_cu_public() * 16u) a.order = nullptr;
  if (a.flags & TC_TRACE_PACKETS) {
    if (T == 64)
      hipLaunchKernelGGL(k_trace_packet<64>, dim3(grid), dim3(64), 0, (hipStream_t)stream, a);
    else if (T == 256)
      hipLaunchKernelGGL(k_trace_packet<256>, dim3(grid), dim3(256), 0, (hipStream_t)stream, a);
    else
      hipLaunchKernelGGL(k_trace_packet<128>, dim3(grid), dim3(128), 0, (hipStream_t)stream, a);
    return hipGetLastError() == hipSuccess ? TC_OK : TC_ERROR_LAUNCH;
  }
  if (T == 64)
    hipLaunchKernelGGL(k_trace<64>, dim3(grid), dim3(64), 0, (hipStream_t)stream, a);
  else if (T == 256)
    hipLaunchKernelGGL(k_trace<256>, dim3(grid), dim3(256), 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL(k_trace<128>, dim3(grid), dim3(128), 0, (hipStream_t)stream, a);
  return hipGetLastError() == hipSuccess ? TC_OK : TC_ERROR_LAUNCH;
}

extern "C" tc_status tc_trace_rays(const tc_bindings* b, tc_config config, const tc_accel* accel, const tc_trace_params* p,
                                   tc_stream stream) {
  return trace_rays(b, config, accel, p, nullptr, stream);
}
