// tc_bvh.h -- BLAS / TLAS build arguments.
#pragma once

#include "tc_sort.h"

namespace tc {

struct BvhArgs {
  tc_scene_building* build;
  const tc_render_instance* instances;
  uint32_t numInstances;
  uint32_t capacity;  // CLAS references the arrays hold
  // BLAS
  uint64_t* keys;  // sort input
  uint32_t* vals;
  const uint64_t* sortedKeys;
  const uint32_t* sortedVals;
  uint64_t* leafAddr;  // CLAS address per sorted position (blasLeaves)
  uint64_t* leafInfo;  // its header's counts | clusterID << 32 (blasLeafInfo)
  // of instances that lie in several chunks of the build, per position
  uint32_t* waitEnd;    // the subtree that ends there and waits for a sibling from outside its chunk, or 0
  uint32_t* waitBegin;  // ... that begins there
  uint64_t* meet;       // the climb that waits at the boundary before it, or 0 (instances of very many chunks)
  tc_bvh_node* nodes;  // blasNodes
  tc_bvh4_node* nodes4;  // blasNodes4
  tc_aabb* nodeBox;    // union box of every internal node
  // TLAS
  tc_tlas_instance* tlasInst;
  tc_aabb* tlasLeafBox;
  uint64_t* tlasKeys;
  uint32_t* tlasVals;
  const uint64_t* tlasSortedKeys;
  const uint32_t* tlasSortedVals;
  uint32_t* tlasChild;
  uint32_t* tlasParent;
  uint32_t* tlasCounter;
  tc_bvh_node* tlasNodes;
  tc_bvh4_node* tlasNodes4;
  tc_aabb* tlasNodeBox;
  uint32_t* tlasRoot;  // [0] root word, [1] instance count
};

struct AccelLayout {
  uint64_t blasNodes, blasLeaves, nodeBox, waitEnd, waitBegin, meet;
  uint64_t blasNodes4, tlasNodes4, blasLeafInfo;
  uint64_t tlasInstances, tlasNodes, tlasNodeBox, tlasLeafBox, tlasChild, tlasParent, tlasCounter, tlasKeys, tlasVals,
      tlasRoot;
  uint64_t total;
};

// 24-bit Morton code (8 bits per axis) of the box centre, normalised to
// [lo, hi]: the BLAS key below the instance, three radix digits
__device__ __forceinline__ uint32_t morton24_of(const float* blo, const float* bhi, const float* lo, const float* hi) {
  uint32_t code = 0;
  for (int k = 0; k < 3; k++) {
    const float c = (blo[k] + bhi[k]) * 0.5f;
    const float ext = hi[k] - lo[k];
    float n = ext > 0.0f ? (c - lo[k]) / ext : 0.5f;
    n = fminf(fmaxf(n, 0.0f), 1.0f);
    uint32_t q = (uint32_t)(n * 255.0f + 0.5f);
    q = (q | (q << 8)) & 0x0300F00Fu;
    q = (q | (q << 4)) & 0x030C30C3u;
    q = (q | (q << 2)) & 0x09249249u;
    code |= q << k;
  }
  return code;
}

AccelLayout accel_layout(uint32_t capacity, uint32_t numInstances);

}  // namespace tc
