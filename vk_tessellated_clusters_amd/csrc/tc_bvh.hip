// tc_bvh.hip -- per-instance BLAS and the TLAS over instances.
//
// Replaces the NV cluster BLAS build and the TLAS update
// (renderer_raytrace_clusters_tess.cpp:695-745, renderer.cpp:318-337):
//   keys    24-bit Morton code (8 bits per axis) of every CLAS centre inside
//           its instance's geometry bounds, the instance index above it:
//           (instance << 32) | morton24, one 64-bit key;
//   sort    the radix sort of tc_sort.hip (one upsweep, then one
//           single-pass launch per digit) over the three Morton digits and
//           the one or two instance digits (stable, CLAS order breaks ties);
//   build   Karras' binary radix tree over each instance's key segment
//           (internal nodes of instance i live at [s_i, s_i + n_i - 1)) with
//           its boxes, from the leaves up, in LDS for subtrees inside one
//           workgroup's chunk of sorted positions; a node's four-wide record is
//           written with it;
//   TLAS    the same builder over the instances' world-space boxes, with a
//           30-bit Morton code (morton_of) per instance.
#include <algorithm>

#include "tc_bvh.h"
#include "tc_insert.h"

namespace tc {

// 30-bit Morton code of the box centre, normalised to [lo, hi]
__host__ __device__ __forceinline__ uint32_t morton_of(const float* blo, const float* bhi, const float* lo,
                                                       const float* hi) {
  uint32_t code = 0;
  for (int k = 0; k < 3; k++) {
    const float c = (blo[k] + bhi[k]) * 0.5f;
    const float ext = hi[k] - lo[k];
    float n = ext > 0.0f ? (c - lo[k]) / ext : 0.5f;
    n = fminf(fmaxf(n, 0.0f), 1.0f);
    uint32_t q = (uint32_t)(n * 1023.0f + 0.5f);
    q = (q | (q << 16)) & 0x030000FFu;
    q = (q | (q << 8)) & 0x0300F00Fu;
    q = (q | (q << 4)) & 0x030C30C3u;
    q = (q | (q << 2)) & 0x09249249u;
    code |= q << k;
  }
  return code;
}

// instance owning global reference position k (lists are contiguous in
// instance order after blas_setup_insertion)
__device__ __forceinline__ uint32_t owner_instance(const tc_blas_build_info* infos, uint32_t numInstances, uint64_t base,
                                                   uint32_t k) {
  uint32_t lo = 0, hi = numInstances;  // last i with start(i) <= k
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) / 2;
    const uint64_t s = (infos[mid].clusterReferences - base) / 8;
    if (s <= k)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// Instances whose list starts a keys workgroup stages in LDS for the owner
// search (more instances search the lists in global memory).
constexpr uint32_t kKeysLdsInstances = 4096;

// BLAS keys over every inserted CLAS reference.  A reference's header loads
// while its owner is searched among the list starts.
__global__ __launch_bounds__(256) void k_blas_keys(BvhArgs a) {
  __shared__ uint32_t s_start[kKeysLdsInstances];
  const tc_scene_building* b = a.build;
  const uint32_t n = min(b->blasClusterCounter, a.capacity);
  const tc_blas_build_info* infos = ptr<const tc_blas_build_info>(b->blasBuildInfos);
  const uint64_t* refs = ptr<const uint64_t>(b->blasClusterAddresses);
  const uint64_t base = b->blasClusterAddresses;
  const bool lds = a.numInstances <= kKeysLdsInstances;
  if (lds)
    for (uint32_t i = threadIdx.x; i < a.numInstances; i += blockDim.x)
      s_start[i] = (uint32_t)((gld(&infos[i].clusterReferences) - base) / 8);
  __syncthreads();
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    const tc_clas_header h = gld_record(ptr<const tc_clas_header>(gld(refs + k)));
    uint32_t inst;
    if (lds) {
      uint32_t lo = 0, hi = a.numInstances;  // last i with start(i) <= k
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (s_start[mid] <= k)
          lo = mid;
        else
          hi = mid;
      }
      inst = lo;
    } else {
      inst = owner_instance(infos, a.numInstances, base, k);
    }
    const tc_render_instance& ri = a.instances[inst];
    const uint32_t m = morton24_of(h.lo, h.hi, ri.geoLo, ri.geoHi);
    a.keys[k] = ((uint64_t)inst << 32) | m;
    a.vals[k] = k;
  }
}

// length of the common prefix of keys i and j (ties broken by index);
// -1 outside [first, last]
__device__ __forceinline__ int delta(const uint64_t* keys, int64_t i, int64_t j, int64_t first, int64_t last) {
  if (j < first || j > last) return -1;
  const uint64_t ki = keys[i], kj = keys[j];
  if (ki == kj) return 64 + __clz((uint32_t)(i ^ j));
  return __clzll(ki ^ kj);
}

// Karras (2012) radix tree for the segment [first, last] of sorted keys;
// thread handles internal node `g` (global index first + local j).
__device__ __forceinline__ void karras_node(const uint64_t* keys, int64_t first, int64_t last, int64_t i, uint32_t* child,
                                            uint32_t* parent, uint32_t leafParentBase) {
  const int d = (delta(keys, i, i + 1, first, last) - delta(keys, i, i - 1, first, last)) >= 0 ? 1 : -1;
  const int dmin = delta(keys, i, i - d, first, last);
  int64_t lmax = 2;
  while (delta(keys, i, i + lmax * d, first, last) > dmin) lmax *= 2;
  int64_t l = 0;
  for (int64_t t = lmax / 2; t >= 1; t /= 2)
    if (delta(keys, i, i + (l + t) * d, first, last) > dmin) l += t;
  const int64_t j = i + l * d;
  const int dnode = delta(keys, i, j, first, last);
  int64_t s = 0;
  int64_t t = l;
  do {
    t = (t + 1) / 2;
    if (delta(keys, i, i + (s + t) * d, first, last) > dnode) s += t;
  } while (t > 1);
  const int64_t gamma = i + s * d + min(d, 0);
  const int64_t lo = min(i, j), hi = max(i, j);
  // children: leaf flag + position relative to `first`, or internal node
  const uint32_t c0 = (lo == gamma) ? (TC_BVH_LEAF | (uint32_t)(gamma - first)) : (uint32_t)(gamma - first);
  const uint32_t c1 = (hi == gamma + 1) ? (TC_BVH_LEAF | (uint32_t)(gamma + 1 - first)) : (uint32_t)(gamma + 1 - first);
  const int64_t node = i - first;
  child[2 * (first + node) + 0] = c0;
  child[2 * (first + node) + 1] = c1;
  // parents (global indices), leaves offset by leafParentBase
  if (c0 & TC_BVH_LEAF)
    parent[leafParentBase + first + (c0 & ~TC_BVH_LEAF)] = (uint32_t)(first + node);
  else
    parent[first + c0] = (uint32_t)(first + node);
  if (c1 & TC_BVH_LEAF)
    parent[leafParentBase + first + (c1 & ~TC_BVH_LEAF)] = (uint32_t)(first + node);
  else
    parent[first + c1] = (uint32_t)(first + node);
}

// segment [first, last] of instance inst in the sorted reference list
__device__ __forceinline__ void blas_segment(const BvhArgs& a, uint32_t inst, uint32_t n, int64_t& first, int64_t& last) {
  const tc_blas_build_info& bi = ptr<const tc_blas_build_info>(a.build->blasBuildInfos)[inst];
  first = (int64_t)((bi.clusterReferences - a.build->blasClusterAddresses) / 8);
  last = first + (int64_t)bi.clusterReferencesCount - 1;
}

// Box of sorted leaf k from its CLAS header; also writes the leaf's info
// word (counts | clusterID << 32) from the same header.  The chunk launch
// stages every leaf once; the leaves of straddling nodes are read again.
__device__ __forceinline__ void leaf_box_at(const BvhArgs& a, uint32_t k, uint64_t addr, float lo[3], float hi[3]) {
  const tc_clas_header h = gld_record(ptr<const tc_clas_header>(addr));
  for (int c = 0; c < 3; c++) lo[c] = h.lo[c], hi[c] = h.hi[c];
  gst(a.leafInfo + k, (uint64_t)h.counts | (uint64_t)h.clusterID << 32);
}
__device__ __forceinline__ void leaf_box(const BvhArgs& a, uint32_t k, float lo[3], float hi[3]) {
  leaf_box_at(a, k, gld(a.leafAddr + k), lo, hi);
}

// One slot of a four-wide record: a box and its child word.
struct Slot4 {
  float lo[3], hi[3];
  uint32_t c;
};
__device__ __forceinline__ Slot4 slot4(const float* lo, const float* hi, uint32_t c) {
  Slot4 r;
  for (int q = 0; q < 3; q++) r.lo[q] = lo[q], r.hi[q] = hi[q];
  r.c = c;
  return r;
}

// Four-wide record of a binary node: its children in order, each internal
// child replaced by that child's two children, empty slots last.  Child 0
// gives a0 (and a1 when internal), child 1 gives b0 (and b1).  The slots
// are chosen by selects, so the record stays in registers.
__device__ __forceinline__ Slot4 sel4(bool c, const Slot4& x, const Slot4& y) {
  Slot4 r;
  for (int q = 0; q < 3; q++) r.lo[q] = c ? x.lo[q] : y.lo[q], r.hi[q] = c ? x.hi[q] : y.hi[q];
  r.c = c ? x.c : y.c;
  return r;
}
__device__ __forceinline__ tc_bvh4_node make4(bool leaf0, const Slot4& a0, const Slot4& a1, bool leaf1, const Slot4& b0,
                                              const Slot4& b1) {
  Slot4 e;
  for (int q = 0; q < 3; q++) e.lo[q] = INFINITY, e.hi[q] = -INFINITY;
  e.c = TC_BVH4_EMPTY;
  const Slot4 s[4] = {a0, sel4(leaf0, b0, a1), sel4(leaf0, sel4(leaf1, e, b1), b0), sel4(leaf0 || leaf1, e, b1)};
  tc_bvh4_node o;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    for (int q = 0; q < 3; q++) o.lo[q][k] = s[k].lo[q], o.hi[q][k] = s[k].hi[q];
    o.child[k] = s[k].c;
  }
  for (int q = 0; q < 4; q++) o._pad[q] = 0;
  return o;
}

// Four-wide record of binary node n of a tree whose node array starts at
// `nodes` (child indices relative to it; its internal children are final).
__device__ __forceinline__ tc_bvh4_node collapse4_of(const tc_bvh_node& n, const tc_bvh_node* nodes) {
  Slot4 g[2][2];
  bool leaf[2];
  for (int c = 0; c < 2; c++) {
    const uint32_t ch = c ? n.child1 : n.child0;
    leaf[c] = (ch & TC_BVH_LEAF) != 0;
    if (leaf[c]) {
      g[c][0] = g[c][1] = slot4(c ? n.lo1 : n.lo0, c ? n.hi1 : n.hi0, ch);
    } else {
      const tc_bvh_node m = gld_record(nodes + ch);
      g[c][0] = slot4(m.lo0, m.hi0, m.child0);
      g[c][1] = slot4(m.lo1, m.hi1, m.child1);
    }
  }
  return make4(leaf[0], g[0][0], g[0][1], leaf[1], g[1][0], g[1][1]);
}
__device__ __forceinline__ void collapse4(const tc_bvh_node* nodes, uint32_t i, tc_bvh4_node* out) {
  gst_record(out + i, collapse4_of(gld_record(nodes + i), nodes));
}

// The tree of every instance and its boxes in two launches, from the leaves up
// (Apetrei 2014) with Karras' (2012) node numbers, and with no device-scope
// fence.
//
// A subtree covers sorted positions [l, r].  Keys l - 1 and l share a prefix of
// some length, and so do keys r and r + 1; the longer of the two says whether
// its sibling begins at r + 1 (it is a left child, node number r) or ends at
// l - 1 (a right child, number l), so the boundary between the two names their
// meeting place.  Of two siblings the second to arrive there makes their
// parent, whose outer prefixes are the siblings'.  No node is searched for.
//
// k_blas_build: a workgroup owns a chunk of kRefitChunk sorted positions, one
// thread per position.  It stages the leaves' boxes (from their CLAS headers,
// which also give the leaf info words) and the prefixes in LDS, the leaves
// climb there, and the binary and four-wide records are written once every
// climb is done.  Subtrees whose sibling reaches out of the chunk, some ten per
// chunk boundary, are noted at their ends for the second launch.
// With Karras' searches in a launch before, 36 bytes a CLAS of topology went
// through memory, and one workgroup of 66 registers filled a CU; both took 67 us
// at 310,000 CLAS in 64 instances, 470 us at 3.3 million, 31 us at 8192 in one,
// with the searches in this launch 48, 360 and 25 us, and now 44, 314 and 18 us:
// 290 bytes a CLAS at 3.0 TB/s at the largest, waits and the records' strided
// stores (a fifth) at the smallest.  Two workgroups of 16 waves share a CU.
//
// k_blas_refit_top: one workgroup per instance that lies in several chunks goes
// on with the climbs.
constexpr uint32_t kRefitChunkBits = 10;
constexpr uint32_t kRefitChunk = 1u << kRefitChunkBits;
constexpr uint32_t kRefitThreads = kRefitChunk;
constexpr uint32_t kRefitTopThreads = 256;
constexpr uint32_t kTopClimbs = 512;  // that meet in LDS
constexpr uint32_t kTopTable = 2 * kTopClimbs;

// Writes internal node `node` from its children's boxes.
__device__ __forceinline__ tc_bvh_node write_node(const BvhArgs& a, uint32_t node, uint32_t c0w, uint32_t c1w,
                                                  const tc_aabb& b0, const tc_aabb& b1) {
  tc_bvh_node out;
  for (int q = 0; q < 3; q++) out.lo0[q] = b0.lo[q], out.hi0[q] = b0.hi[q], out.lo1[q] = b1.lo[q], out.hi1[q] = b1.hi[q];
  out.child0 = c0w;
  out.child1 = c1w;
  out._pad0 = out._pad1 = 0;
  gst_record(a.nodes + node, out);
  return out;
}

// Place of a child's box in the chunk that starts at c0.
__device__ __forceinline__ uint32_t box_at(uint32_t word, uint32_t first, uint32_t c0) {
  return first + (word & ~TC_BVH_LEAF) - c0 + ((word & TC_BVH_LEAF) ? kRefitChunk : 0u);
}

// Length of the common prefix of the keys at positions x and y of one
// instance, plus one: of their Morton codes (the keys' high words are the
// instance), of the positions where the codes are equal.
__device__ __forceinline__ uint32_t key_prefix(uint32_t cx, uint32_t cy, uint32_t x, uint32_t y) {
  const uint32_t v = cx ^ cy;
  return 1u + (v ? __clz(v) : 32u + __clz(x ^ y));
}

// A subtree that waits for a sibling from outside its chunk: its other end,
// from the chunk's start, and the prefix there.
__device__ __forceinline__ uint32_t pack_wait(uint32_t far, uint32_t outer) { return 1u << 31 | outer << 16 | far; }

__global__ __launch_bounds__(kRefitThreads) __attribute__((amdgpu_waves_per_eu(8))) void k_blas_build(BvhArgs a) {
  constexpr uint32_t kNone = ~0u, kDone = ~0u;
  __shared__ tc_aabb s_box[2 * kRefitChunk + 1];  // internal nodes' union boxes, leaves' boxes, an empty one
  __shared__ uint32_t s_child[kRefitChunk][2];
  __shared__ uint32_t s_meet[kRefitChunk + 1];  // per boundary: 0, the subtree that waits there, or kDone
  __shared__ uint8_t s_prefix[kRefitChunk + 4];  // per boundary: key_prefix of its two sides, 0 at an instance's ends
  const tc_scene_building* b = a.build;
  const uint32_t n = min(b->blasClusterCounter, a.capacity);
  const uint64_t* refs = ptr<const uint64_t>(b->blasClusterAddresses);
  const uint32_t j = threadIdx.x;
  if (j == 0)
    for (int q = 0; q < 3; q++) s_box[2 * kRefitChunk].lo[q] = INFINITY, s_box[2 * kRefitChunk].hi[q] = -INFINITY;
  for (uint32_t c0 = blockIdx.x * kRefitChunk; c0 < n; c0 += gridDim.x * kRefitChunk) {
    const uint32_t c1 = min(c0 + kRefitChunk, n), cnt = c1 - c0;
    const uint32_t k = c0 + j;
    uint32_t first = 0, last = 0;
    bool valid = false;
    s_child[j][0] = kNone;
    s_meet[j] = 0;
    if (j == 0) s_meet[kRefitChunk] = 0;
    if (k < c1) {
      const uint64_t key = gld(a.sortedKeys + k), before = gld(a.sortedKeys + (k ? k - 1 : 0u)),
                     after = gld(a.sortedKeys + (k + 1 < n ? k + 1 : k));
      const uint64_t addr = gld(refs + gld(a.sortedVals + k));
      int64_t f, l;
      blas_segment(a, (uint32_t)(key >> 32), n, f, l);
      first = (uint32_t)f, last = (uint32_t)l;
      valid = k >= first && k <= last;
      s_prefix[j] = valid && k != first && before >> 32 == key >> 32
                        ? (uint8_t)key_prefix((uint32_t)before, (uint32_t)key, k - 1, k)
                        : (uint8_t)0;
      if (k + 1 == c1)
        s_prefix[cnt] = valid && k != last && k + 1 < n && after >> 32 == key >> 32
                            ? (uint8_t)key_prefix((uint32_t)key, (uint32_t)after, k, k + 1)
                            : (uint8_t)0;
      gst(a.leafAddr + k, addr);
      float lo[3], hi[3];
      leaf_box_at(a, k, addr, lo, hi);
      for (int q = 0; q < 3; q++) s_box[kRefitChunk + j].lo[q] = lo[q], s_box[kRefitChunk + j].hi[q] = hi[q];
    }
    __syncthreads();
    if (valid && first != last) {  // (a single CLAS is its instance's root)
      uint32_t l = j, r = j;
      while (true) {
        const uint32_t dl = s_prefix[l], dr = s_prefix[r + 1];
        if ((dl | dr) == 0) break;  // the instance's root, written where it was made
        const bool left = dr > dl;
        const uint32_t at = left ? r + 1 : l;
        const uint32_t mine = 1u + (left ? l : r) + (left ? 1u << 16 : 0u);
        if (at == 0 || at == cnt) {  // the sibling lies in another chunk
          s_meet[at] = mine;
          break;
        }
        // the meeting orders LDS only (s_box, s_meet)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        const uint32_t other = atomicExch(&s_meet[at], mine);
        if (other == 0) break;  // first to arrive
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        s_meet[at] = kDone;
        if (left)
          r = (other - 1) & 0xFFFFu;
        else
          l = (other - 1) & 0xFFFFu;
        const uint32_t ul = s_prefix[l], ur = s_prefix[r + 1];
        const bool leaf0 = l + 1 == at, leaf1 = r == at, root = (ul | ur) == 0;
        const tc_aabb &b0 = s_box[at - 1 + (leaf0 ? kRefitChunk : 0u)], &b1 = s_box[at + (leaf1 ? kRefitChunk : 0u)];
        tc_aabb self;
        for (int q = 0; q < 3; q++) self.lo[q] = fminf(b0.lo[q], b1.lo[q]), self.hi[q] = fmaxf(b0.hi[q], b1.hi[q]);
        const uint32_t node = !root && ur > ul ? r : l;
        s_box[node] = self;
        s_child[node][0] = (leaf0 ? TC_BVH_LEAF : 0u) | (c0 + at - 1 - first);
        s_child[node][1] = (leaf1 ? TC_BVH_LEAF : 0u) | (c0 + at - first);
        if (root) gst_record(a.nodeBox + first, self);
      }
    }
    __syncthreads();
    // the subtrees that end or begin at this position and wait for a sibling
    // from outside (an instance inside the chunk has none)
    const uint32_t chunks = (last >> kRefitChunkBits) - (first >> kRefitChunkBits);
    if (valid && chunks != 0) {
      const uint32_t me = s_meet[j + 1], mb = s_meet[j];
      const uint32_t fe = (me - 1) & 0xFFFFu, fb = (mb - 1) & 0xFFFFu;
      gst(a.waitEnd + k, me != 0 && me != kDone && (me - 1) >> 16 != 0 ? pack_wait(fe, s_prefix[fe]) : 0u);
      gst(a.waitBegin + k, mb != 0 && mb != kDone && (mb - 1) >> 16 == 0 ? pack_wait(fb, s_prefix[fb + 1]) : 0u);
      if (chunks > kTopClimbs) gst(a.meet + k, (uint64_t)0);
    }
    // binary and four-wide records of the chunk's internal nodes, one per thread, from LDS (the grandchildren of a local node lie in the
    // chunk): neighbouring threads write neighbouring records, and the climbs,
    // in which few lanes are left after a level or two, store nothing
    if (s_child[j][0] != kNone) {
      const uint32_t cw[2] = {s_child[j][0], s_child[j][1]};
      const uint32_t at[2] = {box_at(cw[0], first, c0), box_at(cw[1], first, c0)};
      write_node(a, k, cw[0], cw[1], s_box[at[0]], s_box[at[1]]);
      // slots as make4 orders them, by their boxes' places: the record leaves
      // a vector at a time, so that the kernel keeps to 64 registers and two
      // workgroups share a CU
      const bool leaf0 = (cw[0] & TC_BVH_LEAF) != 0, leaf1 = (cw[1] & TC_BVH_LEAF) != 0;
      const uint32_t a1w = leaf0 ? 0u : s_child[at[0]][1], b1w = leaf1 ? 0u : s_child[at[1]][1];
      const uint32_t a0w = leaf0 ? cw[0] : s_child[at[0]][0], b0w = leaf1 ? cw[1] : s_child[at[1]][0];
      uint32_t w[4], p[4];
      w[0] = a0w;
      w[1] = leaf0 ? b0w : a1w;
      w[2] = leaf0 ? (leaf1 ? TC_BVH4_EMPTY : b1w) : b0w;
      w[3] = leaf0 || leaf1 ? TC_BVH4_EMPTY : b1w;
#pragma unroll
      for (int q = 0; q < 4; q++) p[q] = w[q] == TC_BVH4_EMPTY ? 2 * kRefitChunk : box_at(w[q], first, c0);
      float* out = reinterpret_cast<float*>(a.nodes4 + k);
#pragma unroll
      for (int q = 0; q < 6; q++) {
        typedef float f4 __attribute__((ext_vector_type(4)));
        const auto side = [&](int i) { return q < 3 ? s_box[p[i]].lo[q % 3] : s_box[p[i]].hi[q % 3]; };
        gst(reinterpret_cast<f4*>(out) + q, f4{side(0), side(1), side(2), side(3)});
      }
      typedef uint32_t u4 __attribute__((ext_vector_type(4)));
      gst(reinterpret_cast<u4*>(out) + 6, u4{w[0], w[1], w[2], w[3]});
      gst(reinterpret_cast<u4*>(out) + 7, u4{0u, 0u, 0u, 0u});
    }
    __syncthreads();
  }
}

// A child of a node being refit: an internal one's binary record (its union is
// the child's box, and its two slots are the grandchildren of the four-wide
// record), or a leaf's box twice.
struct RefitChild {
  Slot4 s[2];
  uint32_t word;
};
__device__ __forceinline__ RefitChild refit_child(const tc_bvh_node& m, uint32_t word) {
  RefitChild r;
  r.s[0] = slot4(m.lo0, m.hi0, m.child0);
  r.s[1] = slot4(m.lo1, m.hi1, m.child1);
  r.word = word;
  return r;
}
// A child that is final before this launch, from memory.
__device__ __forceinline__ RefitChild refit_child_at(const BvhArgs& a, uint32_t first, uint32_t word) {
  RefitChild r;
  if (word & TC_BVH_LEAF) {
    float lo[3], hi[3];
    leaf_box(a, first + (word & ~TC_BVH_LEAF), lo, hi);
    r.s[0] = r.s[1] = slot4(lo, hi, word);
    r.word = word;
  } else {
    r = refit_child(gld_record(a.nodes + first + word), word);
  }
  return r;
}
__device__ __forceinline__ tc_aabb union_box(const Slot4& x, const Slot4& y) {
  tc_aabb b;
  for (int q = 0; q < 3; q++) b.lo[q] = fminf(x.lo[q], y.lo[q]), b.hi[q] = fmaxf(x.hi[q], y.hi[q]);
  return b;
}

// Refit of straddling node `node`: its binary record (returned) and its
// four-wide one.
__device__ __forceinline__ tc_bvh_node refit_top_node(const BvhArgs& a, uint32_t node, uint32_t first, const RefitChild& c0,
                                                      const RefitChild& c1) {
  const tc_bvh_node out =
      write_node(a, node, c0.word, c1.word, union_box(c0.s[0], c0.s[1]), union_box(c1.s[0], c1.s[1]));
  gst_record(a.nodes4 + node,
             make4((c0.word & TC_BVH_LEAF) != 0, c0.s[0], c0.s[1], (c1.word & TC_BVH_LEAF) != 0, c1.s[0], c1.s[1]));
  if (node == first) {  // instance root, read by the TLAS
    tc_aabb self;
    for (int q = 0; q < 3; q++) self.lo[q] = fminf(out.lo0[q], out.lo1[q]), self.hi[q] = fmaxf(out.hi0[q], out.hi1[q]);
    gst_record(a.nodeBox + node, self);
  }
  return out;
}

// TLAS record (written) and world box of instance i.
__device__ __forceinline__ tc_aabb tlas_prep_one(const BvhArgs& a, const float* xforms /* 24 floats per instance */, uint32_t i) {
  const tc_blas_build_info bi = ptr<const tc_blas_build_info>(a.build->blasBuildInfos)[i];
  const uint32_t first = (uint32_t)((bi.clusterReferences - a.build->blasClusterAddresses) / 8);
  const uint32_t cnt = bi.clusterReferencesCount;
  tc_tlas_instance t;
  for (int q = 0; q < 12; q++) t.objectToWorld[q] = xforms[24 * i + q], t.worldToObject[q] = xforms[24 * i + 12 + q];
  t.blasNodes = reinterpret_cast<uint64_t>(a.nodes + first);
  t.blasLeaves = reinterpret_cast<uint64_t>(a.leafAddr + first);
  t.blasRoot = cnt == 1 ? TC_BVH_LEAF : 0u;
  t.numClusters = cnt;
  t.flags = 1;
  t._pad = 0;
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  if (cnt == 1) {
    // a single CLAS is the root and has no parent to refit: its box and info here
    const tc_clas_header h = *ptr<const tc_clas_header>(a.leafAddr[first]);
    for (int q = 0; q < 3; q++) lo[q] = h.lo[q], hi[q] = h.hi[q];
    a.leafInfo[first] = (uint64_t)h.counts | (uint64_t)h.clusterID << 32;
  } else if (cnt > 1) {
    const tc_aabb bx = a.nodeBox[first];
    for (int q = 0; q < 3; q++) lo[q] = bx.lo[q], hi[q] = bx.hi[q];
  }
  a.tlasInst[i] = t;
  // world box of the object box corners
  float wlo[3] = {INFINITY, INFINITY, INFINITY}, whi[3] = {-INFINITY, -INFINITY, -INFINITY};
  if (cnt > 0)
    for (int c = 0; c < 8; c++) {
      const float p[3] = {(c & 1) ? hi[0] : lo[0], (c & 2) ? hi[1] : lo[1], (c & 4) ? hi[2] : lo[2]};
      for (int r = 0; r < 3; r++) {
        const float* m = t.objectToWorld + 4 * r;
        const float w = ((m[0] * p[0] + m[1] * p[1]) + m[2] * p[2]) + m[3];
        wlo[r] = fminf(wlo[r], w);
        whi[r] = fmaxf(whi[r], w);
      }
    }
  // widen by a few ULP-scale steps so rounding of the transformed corners
  // never cuts off a hit found in object space
  tc_aabb wb;
  for (int q = 0; q < 3; q++) {
    const float e = cnt > 0 ? 1e-6f * fmaxf(fmaxf(fabsf(wlo[q]), fabsf(whi[q])), 1e-3f) : 0.0f;
    wb.lo[q] = wlo[q] - e, wb.hi[q] = whi[q] + e;
  }
  return wb;
}

// The climbs of an instance, one from each chunk boundary where the subtrees on
// both sides wait for each other.  Higher up, a sibling is a subtree that waits
// (read with its record ahead of this level's stores: one round trip a level),
// or another climb's: two climbs meet in LDS, where the first leaves its
// record, far end and outer prefix in its slot and the slot's number in a table
// by boundary.  More climbs than kTopClimbs (half a million CLAS in one
// instance) meet in global memory.
// Bound by some 16 levels of a round trip and the stores before it.  64
// instances of up to 130,000 CLAS 42.7 -> 28.6 us, 500 meshes 30 -> 15.5, 5
// instances of 5200 23 -> 15, 64 instances of 51,000 160 -> 122 us.  With a climb
// for every waiting subtree instead, which needs no look-ups, 288 us and 1547 us:
// most lanes of a wave stop at their first meeting.
__device__ __forceinline__ void climb_instance(const BvhArgs& a, uint32_t inst) {
  __shared__ uint32_t s_at[kTopTable];    // boundary, or ~0
  __shared__ uint32_t s_slot[kTopTable];  // 0, or the slot that waits there + 1
  __shared__ __align__(16) tc_bvh_node s_rec[kTopClimbs];  // (_pad0: far end, _pad1: outer prefix)
  const tc_scene_building* b = a.build;
  const uint32_t n = min(b->blasClusterCounter, a.capacity);
  const tc_blas_build_info& bi = ptr<const tc_blas_build_info>(b->blasBuildInfos)[inst];
  if (bi.clusterReferencesCount < 2) return;
  const int64_t first64 = (int64_t)((bi.clusterReferences - b->blasClusterAddresses) / 8);
  if (first64 >= (int64_t)n) return;
  const uint32_t first = (uint32_t)first64, last = min(first + bi.clusterReferencesCount, n) - 1;
  const uint32_t chunk0 = first >> kRefitChunkBits, count = (last >> kRefitChunkBits) - chunk0;
  if (count == 0) return;
  const bool lds = count <= kTopClimbs;
  if (lds)
    for (uint32_t w = threadIdx.x; w < kTopTable; w += kRefitTopThreads) s_at[w] = ~0u, s_slot[w] = 0;
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < count; t += kRefitTopThreads) {
    uint32_t at = (chunk0 + 1 + t) << kRefitChunkBits;
    const uint32_t we = gld(a.waitEnd + at - 1), wb = gld(a.waitBegin + at);
    if (we == 0 || wb == 0) continue;
    uint32_t l = at - kRefitChunk + (we & 0xFFFFu), r = at + (wb & 0xFFFFu);
    uint32_t dl = we >> 16 & 0xFFu, dr = wb >> 16 & 0xFFu;
    RefitChild c0 = refit_child_at(a, first, (l + 1 == at ? TC_BVH_LEAF : 0u) | (at - 1 - first));
    RefitChild c1 = refit_child_at(a, first, (r == at ? TC_BVH_LEAF : 0u) | (at - first));
    while (true) {
      const bool root = (dl | dr) == 0, left = dr > dl;
      const uint32_t node = !root && left ? r : l;  // (the root's l is `first`)
      at = left ? r + 1 : l;
      // the sibling's end there: its node's number, or its leaf
      const uint32_t p = root ? first : (left ? at : at - 1);
      const uint32_t wait = gld((left ? a.waitBegin : a.waitEnd) + p);
      const tc_bvh_node sibRec = gld_record(a.nodes + p);
      const tc_bvh_node made = refit_top_node(a, node, first, c0, c1);
      if (root) break;
      uint32_t far, outer;
      RefitChild sib;
      if (wait != 0) {
        far = (p & ~(kRefitChunk - 1)) + (wait & 0xFFFFu), outer = wait >> 16 & 0xFFu;
        sib = refit_child(sibRec, p - first);
        if (far == p) sib = refit_child_at(a, first, TC_BVH_LEAF | (p - first));
      } else if (lds) {
        uint32_t h = (at * 2654435761u) >> (32 - 10);
        static_assert(kTopTable == 1u << 10, "the hash's bits");
        while (true) {  // at most kTopClimbs - 1 boundaries
          const uint32_t seen = atomicCAS(&s_at[h], ~0u, at);
          if (seen == ~0u || seen == at) break;
          h = (h + 1) & (kTopTable - 1);
        }
        // the climb's own slot: it stays in place once the climb stops
        tc_bvh_node own = made;
        own._pad0 = left ? l : r, own._pad1 = left ? dl : dr;
        s_rec[t] = own;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        const uint32_t met = atomicExch(&s_slot[h], t + 1);
        if (met == 0) break;  // first to arrive
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        const tc_bvh_node rec = s_rec[met - 1];
        far = rec._pad0, outer = rec._pad1;
        sib = refit_child(rec, p - first);
      } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        const uint64_t met = atomicExch(reinterpret_cast<unsigned long long*>(a.meet + at),
                                        1ull << 63 | (unsigned long long)(left ? dl : dr) << 32 | (left ? l : r));
        if (met == 0) break;  // first to arrive
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        far = (uint32_t)met, outer = (uint32_t)(met >> 32) & 0xFFu;
        sib = refit_child_at(a, first, p - first);  // (a climb's subtree is no leaf)
      }
      const RefitChild mine = refit_child(made, node - first);
      c0 = left ? mine : sib, c1 = left ? sib : mine;
      if (left)
        r = far, dr = outer;
      else
        l = far, dl = outer;
    }
  }
}

// The climbs; a single instance's workgroup also writes the TLAS, which is that
// instance alone.  Its launch would cost more than its work: frames of one
// instance 208.9 -> 206.4 us (320 x 180), 406.4 -> 402.7 us (1280 x 720); depth
// step on 512^2 rays 343.0 -> 339.8 us.
__global__ __launch_bounds__(kRefitTopThreads) void k_blas_refit_top(BvhArgs a, const float* xforms) {
  if (blockIdx.x >= a.numInstances) return;
  climb_instance(a, blockIdx.x);
  if (a.numInstances != 1) return;
  __syncthreads();
  if (threadIdx.x == 0) {
    tlas_prep_one(a, xforms, 0);
    a.tlasRoot[0] = TC_BVH_LEAF;
    a.tlasRoot[1] = 1;
  }
}

// Per-instance TLAS records and world boxes (one thread per instance).
__global__ void k_tlas_prep(BvhArgs a, const float* xforms) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < a.numInstances) a.tlasLeafBox[i] = tlas_prep_one(a, xforms, i);
}

// Scene bounds and TLAS keys over instances (one workgroup).
__global__ __launch_bounds__(256) void k_tlas_keys(BvhArgs a) {
  __shared__ float s_lo[3][256], s_hi[3][256];
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (uint32_t i = threadIdx.x; i < a.numInstances; i += blockDim.x) {
    const tc_aabb bx = a.tlasLeafBox[i];
    if (!(bx.lo[0] <= bx.hi[0])) continue;
    for (int q = 0; q < 3; q++) lo[q] = fminf(lo[q], (bx.lo[q] + bx.hi[q]) * 0.5f), hi[q] = fmaxf(hi[q], (bx.lo[q] + bx.hi[q]) * 0.5f);
  }
  for (int q = 0; q < 3; q++) s_lo[q][threadIdx.x] = lo[q], s_hi[q][threadIdx.x] = hi[q];
  __syncthreads();
  for (uint32_t s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s)
      for (int q = 0; q < 3; q++) {
        s_lo[q][threadIdx.x] = fminf(s_lo[q][threadIdx.x], s_lo[q][threadIdx.x + s]);
        s_hi[q][threadIdx.x] = fmaxf(s_hi[q][threadIdx.x], s_hi[q][threadIdx.x + s]);
      }
    __syncthreads();
  }
  const float slo[3] = {s_lo[0][0], s_lo[1][0], s_lo[2][0]}, shi[3] = {s_hi[0][0], s_hi[1][0], s_hi[2][0]};
  for (uint32_t i = threadIdx.x; i < a.numInstances; i += blockDim.x) {
    const tc_aabb bx = a.tlasLeafBox[i];
    const bool empty = !(bx.lo[0] <= bx.hi[0]);
    // empty instances sort last and are never entered
    a.tlasKeys[i] = empty ? (0xFFFFFFFFull << 32) | i : ((uint64_t)morton_of(bx.lo, bx.hi, slo, shi) << 32) | i;
    a.tlasVals[i] = i;
  }
}

// TLAS over the (sorted) instances: one thread per sorted position.
__global__ void k_tlas_hierarchy(BvhArgs a) {
  const uint32_t n = a.numInstances;
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    a.tlasCounter[k] = 0;
    if (k + 1 < n) karras_node(a.tlasSortedKeys, 0, (int64_t)n - 1, k, a.tlasChild, a.tlasParent, n);
  }
}

// Bottom-up refit from sorted TLAS leaf k: the second arrival at a node
// writes it.  With WORKGROUP every climber is in one workgroup, so
// workgroup-scope ordering suffices (a device-scope release writes back the
// XCD's L2 at every level).
template <bool WORKGROUP>
__device__ void tlas_refit_leaf(const BvhArgs& a, uint32_t k) {
  const uint32_t n = a.numInstances;
  {
    uint32_t node = a.tlasParent[n + k];
    while (true) {
      if (WORKGROUP)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      else
        __threadfence();
      if (atomicAdd(&a.tlasCounter[node], 1u) == 0) break;
      if (WORKGROUP)
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      else
        __threadfence();
      tc_bvh_node out;
      float lo[2][3], hi[2][3];
      for (int c = 0; c < 2; c++) {
        const uint32_t ch = a.tlasChild[2 * node + c];
        tc_aabb bx = (ch & TC_BVH_LEAF) ? a.tlasLeafBox[a.tlasSortedVals[ch & ~TC_BVH_LEAF]] : a.tlasNodeBox[ch];
        for (int q = 0; q < 3; q++) lo[c][q] = bx.lo[q], hi[c][q] = bx.hi[q];
      }
      for (int q = 0; q < 3; q++) out.lo0[q] = lo[0][q], out.hi0[q] = hi[0][q], out.lo1[q] = lo[1][q], out.hi1[q] = hi[1][q];
      const uint32_t c0 = a.tlasChild[2 * node], c1 = a.tlasChild[2 * node + 1];
      // leaves of the TLAS name instances directly
      out.child0 = (c0 & TC_BVH_LEAF) ? (TC_BVH_LEAF | a.tlasSortedVals[c0 & ~TC_BVH_LEAF]) : c0;
      out.child1 = (c1 & TC_BVH_LEAF) ? (TC_BVH_LEAF | a.tlasSortedVals[c1 & ~TC_BVH_LEAF]) : c1;
      out._pad0 = out._pad1 = 0;
      a.tlasNodes[node] = out;
      tc_aabb self;
      for (int q = 0; q < 3; q++) self.lo[q] = fminf(lo[0][q], lo[1][q]), self.hi[q] = fmaxf(hi[0][q], hi[1][q]);
      a.tlasNodeBox[node] = self;
      if (node == 0) break;
      node = a.tlasParent[node];
    }
  }
}

__global__ void k_tlas_refit(BvhArgs a) {
  const uint32_t n = a.numInstances;
  if (n == 1) return;
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) tlas_refit_leaf<false>(a, k);
}

__global__ void k_tlas_collapse4(BvhArgs a) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i + 1 < a.numInstances) collapse4(a.tlasNodes, i, a.tlasNodes4);
}

// instances the one-workgroup TLAS build (k_tlas_build_small) takes
constexpr uint32_t kTlasRankSort = 1024;

// TLAS root word (internal node 0) and the TLAS element count read by the sort
__global__ void k_tlas_root(BvhArgs a) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    a.tlasRoot[0] = 0;
    a.tlasRoot[1] = a.numInstances;
  }
}

// The whole TLAS in one workgroup for 2 to kTlasRankSort instances, one
// thread per instance: records and world boxes, scene bounds and keys, the
// rank sort, the tree with its boxes from the leaves up (as k_blas_build), and
// the binary and four-wide records.  One workgroup's chain of waits: of 28.8 us
// at 500 instances the ranks took 6.9 (a key of LDS after another), Karras'
// searches 4.0, the climbs with their record stores 6.8, reading the boxes back
// 1.9.  Every thread now ranks four keys at a time, with several threads to an
// instance where there are fewer than half as many as threads: 500 instances
// 29.9 -> 24.3 us, 64 14.5 -> 9.5, 20 10.9 -> 7.3, 8 9.4 -> 6.8.
__global__ __launch_bounds__(kTlasRankSort) void k_tlas_build_small(BvhArgs a, const float* xforms) {
  __shared__ float s_b[6][kTlasRankSort / kWave];
  __shared__ __align__(16) uint64_t s_key[kTlasRankSort + 4];
  __shared__ uint64_t s_sorted[kTlasRankSort];
  __shared__ uint32_t s_rank[kTlasRankSort], s_val[kTlasRankSort];
  __shared__ uint32_t s_child[kTlasRankSort][2], s_meet[kTlasRankSort];
  __shared__ uint8_t s_prefix[kTlasRankSort + 4];
  __shared__ tc_aabb s_leaf[kTlasRankSort], s_box[kTlasRankSort];  // by sorted position, by internal node
  const uint32_t n = a.numInstances, i = threadIdx.x, lane = lane_id(), wave = threadIdx.x / kWave;
  tc_aabb bx;
  bool empty = true;
  float c[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  if (i < n) {
    bx = tlas_prep_one(a, xforms, i);
    empty = !(bx.lo[0] <= bx.hi[0]);
    if (!empty)
      for (int q = 0; q < 3; q++) c[q] = c[3 + q] = (bx.lo[q] + bx.hi[q]) * 0.5f;
  }
  if (i == 0) {
    a.tlasRoot[0] = 0;
    a.tlasRoot[1] = n;
  }
  s_rank[i] = 0;
  s_meet[i] = 0;
  // scene bounds of the instance box centres (k_tlas_keys)
#pragma unroll
  for (int q = 0; q < 3; q++) {
    for (int d = 1; d < kWave; d <<= 1) {
      c[q] = fminf(c[q], __shfl_xor(c[q], d, kWave));
      c[3 + q] = fmaxf(c[3 + q], __shfl_xor(c[3 + q], d, kWave));
    }
  }
  if (lane == 0)
    for (int q = 0; q < 6; q++) s_b[q][wave] = c[q];
  __syncthreads();
  float slo[3] = {INFINITY, INFINITY, INFINITY}, shi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (uint32_t w = 0; w < kTlasRankSort / kWave; w++)
    for (int q = 0; q < 3; q++) slo[q] = fminf(slo[q], s_b[q][w]), shi[q] = fmaxf(shi[q], s_b[3 + q][w]);
  // keys (empty instances sort last and are never entered), then ranks
  if (i < n) s_key[i] = empty ? (0xFFFFFFFFull << 32) | i : ((uint64_t)morton_of(bx.lo, bx.hi, slo, shi) << 32) | i;
  if (i < 4) s_key[n + i] = ~0ull;  // above every key
  __syncthreads();
  {
    // thread i ranks key i % span among its share of the keys
    uint32_t span = kWave;
    while (span < n) span *= 2;
    const uint32_t me = i % span, share = ((n + kTlasRankSort / span - 1) / (kTlasRankSort / span) + 3u) & ~3u;
    const uint32_t j0 = i / span * share, j1 = min(j0 + share, (n + 3u) & ~3u);
    if (me < n && j0 < j1) {
      const uint64_t k = s_key[me];
      uint32_t rank = 0;
      for (uint32_t j = j0; j < j1; j += 4) {
        const ulonglong2 x = *reinterpret_cast<const ulonglong2*>(s_key + j), y = *reinterpret_cast<const ulonglong2*>(s_key + j + 2);
        rank += (x.x < k ? 1u : 0u) + (x.y < k ? 1u : 0u) + (y.x < k ? 1u : 0u) + (y.y < k ? 1u : 0u);
      }
      atomicAdd(&s_rank[me], rank);
    }
  }
  __syncthreads();
  if (i < n) {
    const uint32_t rank = s_rank[i];
    const uint64_t k = s_key[i];
    s_sorted[rank] = k;
    s_val[rank] = i;
    s_leaf[rank] = bx;
  }
  __syncthreads();
  if (i < n) {
    s_prefix[i] = i ? (uint8_t)(1 + __clzll(s_sorted[i - 1] ^ s_sorted[i])) : (uint8_t)0;
    if (i + 1 == n) s_prefix[n] = 0;
  }
  __syncthreads();
  const auto box_of = [&](uint32_t w) -> const tc_aabb& { return (w & TC_BVH_LEAF) ? s_leaf[w & ~TC_BVH_LEAF] : s_box[w]; };
  if (i < n) {
    uint32_t l = i, r = i;
    while (true) {
      const uint32_t dl = s_prefix[l], dr = s_prefix[r + 1];
      if ((dl | dr) == 0) break;  // the root (or the only instance)
      const bool left = dr > dl;
      const uint32_t at = left ? r + 1 : l;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      const uint32_t other = atomicExch(&s_meet[at], 1u + (left ? l : r));
      if (other == 0) break;  // first to arrive
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
      if (left)
        r = other - 1;
      else
        l = other - 1;
      const uint32_t ul = s_prefix[l], ur = s_prefix[r + 1];
      const uint32_t w0 = (l + 1 == at ? TC_BVH_LEAF : 0u) | (at - 1), w1 = (r == at ? TC_BVH_LEAF : 0u) | at;
      const tc_aabb &b0 = box_of(w0), &b1 = box_of(w1);
      tc_aabb self;
      for (int q = 0; q < 3; q++) self.lo[q] = fminf(b0.lo[q], b1.lo[q]), self.hi[q] = fmaxf(b0.hi[q], b1.hi[q]);
      const uint32_t node = ur > ul ? r : l;  // (the root's l is 0)
      s_box[node] = self;
      s_child[node][0] = w0, s_child[node][1] = w1;
    }
  }
  __syncthreads();
  if (i + 1 < n) {
    // a TLAS leaf names its instance: the sorted position's value
    const auto leaf_word = [&](uint32_t w) { return (w & TC_BVH_LEAF) ? (TC_BVH_LEAF | s_val[w & ~TC_BVH_LEAF]) : w; };
    const uint32_t cw[2] = {s_child[i][0], s_child[i][1]};
    const tc_aabb &b0 = box_of(cw[0]), &b1 = box_of(cw[1]);
    tc_bvh_node out;
    for (int q = 0; q < 3; q++) out.lo0[q] = b0.lo[q], out.hi0[q] = b0.hi[q], out.lo1[q] = b1.lo[q], out.hi1[q] = b1.hi[q];
    out.child0 = leaf_word(cw[0]);
    out.child1 = leaf_word(cw[1]);
    out._pad0 = out._pad1 = 0;
    gst_record(a.tlasNodes + i, out);
    Slot4 gs[2][2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if (cw[c] & TC_BVH_LEAF) {
        const tc_aabb& bx = box_of(cw[c]);
        gs[c][0] = gs[c][1] = slot4(bx.lo, bx.hi, leaf_word(cw[c]));
      } else {
#pragma unroll
        for (int d = 0; d < 2; d++) {
          const uint32_t gw = s_child[cw[c]][d];
          const tc_aabb& bx = box_of(gw);
          gs[c][d] = slot4(bx.lo, bx.hi, leaf_word(gw));
        }
      }
    }
    gst_record(a.tlasNodes4 + i, make4((cw[0] & TC_BVH_LEAF) != 0, gs[0][0], gs[0][1], (cw[1] & TC_BVH_LEAF) != 0,
                                       gs[1][0], gs[1][1]));
  }
}

}  // namespace tc

// ------------------------------------------------------------ host entry

namespace tc {

static uint64_t a256(uint64_t v) { return (v + 255) & ~255ull; }

AccelLayout accel_layout(uint32_t capacity, uint32_t numInstances) {
  AccelLayout L{};
  uint64_t o = 0;
  auto put = [&](uint64_t& f, uint64_t bytes) {
    f = o;
    o = a256(o + bytes);
  };
  const uint64_t c = capacity, n = std::max(numInstances, 1u);
  put(L.blasNodes, c * sizeof(tc_bvh_node));
  put(L.blasNodes4, c * sizeof(tc_bvh4_node));
  put(L.blasLeaves, c * 8);
  put(L.blasLeafInfo, c * 8);
  put(L.nodeBox, c * sizeof(tc_aabb));
  put(L.waitEnd, c * 4);
  put(L.waitBegin, c * 4);
  put(L.meet, c * 8);
  put(L.tlasInstances, n * sizeof(tc_tlas_instance));
  put(L.tlasNodes, n * sizeof(tc_bvh_node));
  put(L.tlasNodes4, n * sizeof(tc_bvh4_node));
  put(L.tlasNodeBox, n * sizeof(tc_aabb));
  put(L.tlasLeafBox, n * sizeof(tc_aabb));
  put(L.tlasChild, 2 * n * 4);
  put(L.tlasParent, 2 * n * 4);
  put(L.tlasCounter, n * 4);
  put(L.tlasKeys, n * 8);
  put(L.tlasVals, n * 4);
  put(L.tlasRoot, 256);
  L.total = o;
  return L;
}

}  // namespace tc

using namespace tc;

extern "C" {

uint64_t tc_accel_size(uint32_t capacity, uint32_t numInstances) { return accel_layout(capacity, numInstances).total; }

tc_status tc_accel_bind(void* memory, uint64_t bytes, uint32_t capacity, uint32_t numInstances, tc_accel* out) {
  if (!memory || !out || !capacity || !numInstances) return TC_ERROR_INVALID_ARGUMENT;
  AccelLayout L = accel_layout(capacity, numInstances);
  if (bytes < L.total) return TC_ERROR_INVALID_ARGUMENT;
  char* m = static_cast<char*>(memory);
  out->blasNodes = reinterpret_cast<tc_bvh_node*>(m + L.blasNodes);
  out->blasLeaves = reinterpret_cast<uint64_t*>(m + L.blasLeaves);
  out->tlasInstances = reinterpret_cast<tc_tlas_instance*>(m + L.tlasInstances);
  out->tlasNodes = reinterpret_cast<tc_bvh_node*>(m + L.tlasNodes);
  out->tlasRoot = reinterpret_cast<uint32_t*>(m + L.tlasRoot);
  out->blasNodes4 = reinterpret_cast<tc_bvh4_node*>(m + L.blasNodes4);
  out->tlasNodes4 = reinterpret_cast<tc_bvh4_node*>(m + L.tlasNodes4);
  out->blasLeafInfo = reinterpret_cast<uint64_t*>(m + L.blasLeafInfo);
  out->numInstances = numInstances;
  out->capacity = capacity;
  out->memory = memory;
  out->memoryBytes = bytes;
  return TC_OK;
}

}  // extern "C"

// `inserted`: the keys and the digit counts are those insert_clusters left.
static tc_status accel_build(const tc_bindings* b, tc_config config, const tc_accel* accel, const float* instanceXforms,
                             tc_stream stream, bool inserted) {
  KArgs ka;
  tc_status s = make_args_public(b, config, ka);
  if (s != TC_OK) return s;
  if (!accel || !accel->memory || !instanceXforms || accel->numInstances != b->numRenderInstances) return TC_ERROR_INVALID_ARGUMENT;
  const uint32_t capacity = accel->capacity;
  if (capacity < config.maxGeneratedClusters) return TC_ERROR_INVALID_ARGUMENT;
  AccelLayout L = accel_layout(capacity, accel->numInstances);
  if (accel->memoryBytes < L.total) return TC_ERROR_INVALID_ARGUMENT;
  WsLayout W = ws_layout(config, b->numRenderInstances);
  if (W.sortCapacity < capacity) return TC_ERROR_INVALID_ARGUMENT;
  char* m = static_cast<char*>(accel->memory);
  char* w = static_cast<char*>(b->workspace);
  hipStream_t st = (hipStream_t)stream;

  BvhArgs a;
  a.build = b->build;
  a.instances = b->instances;
  a.numInstances = b->numRenderInstances;
  a.capacity = capacity;
  SortBuffers sb;
  for (int i = 0; i < 2; i++) {
    sb.keys[i] = reinterpret_cast<uint64_t*>(w + W.sortKeys[i]);
    sb.vals[i] = reinterpret_cast<uint32_t*>(w + W.sortVals[i]);
  }
  sb.status = reinterpret_cast<uint64_t*>(w + W.sortStatus);
  sb.state = reinterpret_cast<SortState*>(w + W.sortState);
  sb.capacity = W.sortCapacity;
  sb.maxTiles = W.sortMaxTiles;
  a.keys = sb.keys[0];
  a.vals = sb.vals[0];
  a.leafAddr = reinterpret_cast<uint64_t*>(m + L.blasLeaves);
  a.leafInfo = reinterpret_cast<uint64_t*>(m + L.blasLeafInfo);
  a.waitEnd = reinterpret_cast<uint32_t*>(m + L.waitEnd);
  a.waitBegin = reinterpret_cast<uint32_t*>(m + L.waitBegin);
  a.meet = reinterpret_cast<uint64_t*>(m + L.meet);
  a.nodes = reinterpret_cast<tc_bvh_node*>(m + L.blasNodes);
  a.nodes4 = reinterpret_cast<tc_bvh4_node*>(m + L.blasNodes4);
  a.nodeBox = reinterpret_cast<tc_aabb*>(m + L.nodeBox);
  a.tlasInst = reinterpret_cast<tc_tlas_instance*>(m + L.tlasInstances);
  a.tlasNodes = reinterpret_cast<tc_bvh_node*>(m + L.tlasNodes);
  a.tlasNodes4 = reinterpret_cast<tc_bvh4_node*>(m + L.tlasNodes4);
  a.tlasNodeBox = reinterpret_cast<tc_aabb*>(m + L.tlasNodeBox);
  a.tlasLeafBox = reinterpret_cast<tc_aabb*>(m + L.tlasLeafBox);
  a.tlasChild = reinterpret_cast<uint32_t*>(m + L.tlasChild);
  a.tlasParent = reinterpret_cast<uint32_t*>(m + L.tlasParent);
  a.tlasCounter = reinterpret_cast<uint32_t*>(m + L.tlasCounter);
  a.tlasRoot = reinterpret_cast<uint32_t*>(m + L.tlasRoot);

  const uint32_t grid = std::min<uint32_t>((capacity + 255) / 256, (uint32_t)num_cu_public() * tuning_snapshot().bvhBlocksPerCU);
  // BLAS: keys, sort by (instance, Morton), trees and boxes
  if (!inserted) hipLaunchKernelGGL(k_blas_keys, dim3(grid), dim3(256), 0, st, a);
  uint32_t res = 0;
  // digits 0-2: the 24-bit Morton code; digits 4-5: the instance, where there
  // is more than one
  const InsertPlan ip = insert_plan(b, config);
  radix_sort_digits(sb, &b->build->blasClusterCounter, 0x7u | ((1u << ip.instancePasses) - 1u) << 4, st, &res,
                    inserted ? ip.insertPasses : 0);
  a.sortedKeys = sb.keys[res];
  a.sortedVals = sb.vals[res];
  hipLaunchKernelGGL(k_blas_build, dim3(std::min<uint32_t>((capacity + kRefitChunk - 1) / kRefitChunk, (uint32_t)num_cu_public() * 4)),
                     dim3(kRefitThreads), 0, st, a);
  hipLaunchKernelGGL(k_blas_refit_top, dim3(a.numInstances), dim3(kRefitTopThreads), 0, st, a, instanceXforms);
  if (a.numInstances == 1) return hipGetLastError() == hipSuccess ? TC_OK : TC_ERROR_LAUNCH;
  // TLAS over instances, with key and value arrays of its own
  a.tlasKeys = reinterpret_cast<uint64_t*>(m + L.tlasKeys);
  a.tlasVals = reinterpret_cast<uint32_t*>(m + L.tlasVals);
  if (a.numInstances <= kTlasRankSort) {
    hipLaunchKernelGGL(k_tlas_build_small, dim3(1), dim3(kTlasRankSort), 0, st, a, instanceXforms);
    return hipGetLastError() == hipSuccess ? TC_OK : TC_ERROR_LAUNCH;
  }
  hipLaunchKernelGGL(k_tlas_prep, dim3((a.numInstances + 63) / 64), dim3(64), 0, st, a, instanceXforms);
  hipLaunchKernelGGL(k_tlas_keys, dim3(1), dim3(256), 0, st, a);
  // the TLAS sort's scratch slot is the TLAS child / parent arrays, written
  // only afterwards (32 key bits = 4 passes, so the result lands back in
  // slot 0); it shares the workspace sort state and status words, which
  // hold kMaxInstances keys' tiles
  SortBuffers tb = sb;
  tb.keys[0] = a.tlasKeys;
  tb.vals[0] = a.tlasVals;
  tb.keys[1] = reinterpret_cast<uint64_t*>(m + L.tlasChild);
  tb.vals[1] = reinterpret_cast<uint32_t*>(m + L.tlasParent);
  tb.capacity = a.numInstances;
  hipLaunchKernelGGL(k_tlas_root, dim3(1), dim3(64), 0, st, a);
  uint32_t tres = 0;
  radix_sort_pairs(tb, a.tlasRoot + 1, 32, 32, st, &tres);
  a.tlasSortedKeys = tb.keys[tres];
  a.tlasSortedVals = tb.vals[tres];
  const uint32_t tgrid = (a.numInstances + 255) / 256;
  hipLaunchKernelGGL(k_tlas_hierarchy, dim3(tgrid), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_tlas_refit, dim3(tgrid), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_tlas_collapse4, dim3(tgrid), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? TC_OK : TC_ERROR_LAUNCH;
}

tc_status tc::accel_build_inserted(const tc_bindings* b, tc_config config, const tc_accel* accel, const float* instanceXforms,
                                   tc_stream stream) {
  return accel_build(b, config, accel, instanceXforms, stream, true);
}

extern "C" tc_status tc_accel_build(const tc_bindings* b, tc_config config, const tc_accel* accel, const float* instanceXforms,
                                    tc_stream stream) {
  return accel_build(b, config, accel, instanceXforms, stream, false);
}
