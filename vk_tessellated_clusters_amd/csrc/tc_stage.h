// tc_stage.h -- helpers shared by the stage kernels.
#pragma once

#include "tc_kernels.h"

namespace tc {

enum Stage : uint32_t { kStageClassify = 0, kStageSplit = 1, kStageInstantiate = 2 };

constexpr uint32_t kClassifyWaves = 4;   // waves per classify workgroup
constexpr uint32_t kClassifyTile = 64;   // visible clusters per classify tile, at most
// A tile's four waves take its clusters one after another, so a frame with
// fewer clusters than fill the chip 64 at a time takes smaller tiles: halved
// down to 8 while that leaves fewer than kClassifyTiles tiles.  64 clusters of
// 81 vertices: 72 us in one tile of 64, 21 us in eight of 8; 245 clusters with
// ripple 62 -> 30 us.  Tiles of 4, and 256 or 1024 tiles, measure the same; 2048
// tiles (of 32, at 65,536 clusters) make the frame 1082 -> 1120 us.
constexpr uint32_t kClassifyMinTile = 8;
constexpr uint32_t kClassifyTiles = 512;
constexpr uint32_t kVertCache = 128;     // vertices per wave a classify cluster caches
constexpr uint32_t kInstWaves = 4;       // waves per instantiate workgroup
constexpr uint32_t kInstTile = kInstWaves * 4 * 64;  // part triangles per instantiate tile (4 per lane)

__device__ __forceinline__ ViewParams view_params(const KArgs& a) {
  ViewParams vp;
  vp.eye = mk(a.build->viewPos[0], a.build->viewPos[1], a.build->viewPos[2]);
  vp.nearPlane = a.view->nearPlane;
  vp.vpy = a.view->viewportf[1];
  vp.rate = a.view->tessRate;
  return vp;
}

__device__ __forceinline__ bool has_disp(const KArgs& a, int32_t idx) {
  return (a.cfg.flags & TC_FLAG_DISPLACEMENT) && idx >= 0 && (uint32_t)idx < a.numTextures;
}

// The frame's displacement scale and offset, read once per kernel: vertex
// loops store through pointers the compiler cannot tell apart from the
// frame constants, so a read inside the loop is repeated every iteration.
struct DispGlobal {
  float scale, offset;
};
__device__ __forceinline__ DispGlobal disp_global(const KArgs& a) {
  return DispGlobal{a.view->displacementScale, a.view->displacementOffset};
}

// cluster_classify.comp.glsl:477-479
__device__ __forceinline__ float displaced_height(const DispGlobal& g, const tc_displacement_texture& tex, float scale,
                                                  float offset, v2 uv) {
  float h = sample_height(tex, uv.x, uv.y);
  return (((h * scale) * g.scale) + offset) + g.offset;
}
__device__ __forceinline__ float displaced_height(const KArgs& a, const tc_displacement_texture& tex, float scale,
                                                  float offset, v2 uv) {
  return displaced_height(disp_global(a), tex, scale, offset, uv);
}

// Records how generated vertex `index` was displaced (tc_vertex_tape).
__device__ __forceinline__ void write_tape(const KArgs& a, uint64_t index, v3 base, v3 normal, v2 uv, float scale,
                                           float offset, uint32_t texture) {
  float4* t = reinterpret_cast<float4*>(a.tape + index);
  t[0] = make_float4(base.x, base.y, base.z, normal.x);
  t[1] = make_float4(normal.y, normal.z, uv.x, uv.y);
  t[2] = make_float4(scale * a.view->displacementScale, offset + a.view->displacementOffset, __uint_as_float(texture), 0.0f);
}

// Bytes of our CLAS block for nt triangles and nv vertices (tc_clas_size).
__host__ __device__ constexpr uint32_t clas_block_size(uint32_t nt, uint32_t nv) {
  return (uint32_t)sizeof(tc_clas_header) + ((((nt + TC_CLAS_GROUP_TRIANGLES - 1) / TC_CLAS_GROUP_TRIANGLES) * 24u + 15u) & ~15u) +
         ((nt * 4u + 15u) & ~15u) + ((nv * 12u + 15u) & ~15u);
}

// CLAS bytes reserved per 2X mini batch: the worst case of the batch
// (:732-733 reserves basicClusterSizes[miniBatchTriangles])
constexpr uint32_t kMiniDataSize = clas_block_size(kMiniBatchTris, kMiniBatchVerts);

__device__ __forceinline__ uint64_t max_data_bytes(const tc_config& c) {
  return (uint64_t)c.maxGeneratedClusterMegs * 1024ull * 1024ull;
}

// Last index j of the non-decreasing s_start[0..N) with s_start[j] <= t (0
// when there is none), as a count in two rounds of independent LDS reads:
// the group of eight holding j from every eighth entry, then j within it.
template <uint32_t N>
__device__ __forceinline__ uint32_t find_owner_n(const uint32_t* s_start, uint32_t t) {
  static_assert(N % 8 == 0 && N >= 16, "groups of eight");
  uint32_t g = 0;
#pragma unroll
  for (uint32_t j = 1; j < N / 8; j++) g += s_start[8 * j] <= t ? 1u : 0u;
  const uint32_t* s = s_start + 8 * g;
  uint32_t k = 0;
#pragma unroll
  for (uint32_t i = 1; i < 8; i++) k += s[i] <= t ? 1u : 0u;
  return 8 * g + k;
}
__device__ __forceinline__ uint32_t find_owner(const uint32_t* s_start, uint32_t t) { return find_owner_n<64>(s_start, t); }

// Adds `count` of every active lane to infos[instance].clusterReferencesCount
// with one atomic per distinct instance in the wave (neighbouring lanes
// usually share the instance).
__device__ __forceinline__ void add_blas_reference_counts(tc_blas_build_info* infos, uint32_t key, uint32_t count,
                                                          bool active) {
  uint64_t pending = ballot(active && count != 0);
  while (pending) {
    const uint32_t leader = (uint32_t)__builtin_ctzll(pending);
    const uint32_t lkey = shfl(key, leader);
    const bool same = ((pending >> lane_id()) & 1ull) && key == lkey;
    const uint64_t sameMask = ballot(same);
    const uint32_t sum = wave_sum(same ? count : 0u);
    if (lane_id() == leader) atomicAdd(&infos[lkey].clusterReferencesCount, sum);
    pending &= ~sameMask;
  }
}

// Parts that are instantiated: the accepted prefix of the list.  With
// transient builds (build_setup.comp.glsl:240-253) x + y + 2 <=
// MAX_PART_TRIANGLES of the lower counter x.
__device__ __forceinline__ uint32_t accepted_parts(const KArgs& a) {
  uint32_t cap = a.cfg.maxPartTriangles;
  if (transient_builds(a.cfg.flags)) {
    const uint32_t y = (uint32_t)(a.build->dualPartTriangleCounter >> 32);
    cap = cap > y + 1 ? cap - y - 1 : 0u;
  }
  return min(a.build->partTriangleCounter, cap);
}

// build_setup.comp.glsl:102-264 (transient builds with TC_FLAG_1X_TRANSIENT
// or TC_FLAG_2X_TRANSIENT).  One thread.
__device__ __forceinline__ void build_setup_one(const KArgs& a, int mode) {
  tc_scene_building* b = a.build;
  tc_readback* rb = a.readback;
  const tc_config& cfg = a.cfg;
  if (mode == TC_BUILD_SETUP_CLASSIFY) {
    uint32_t counter = b->visibleClusterCounter;
    rb->numVisibleClusters = counter;
    counter = min(counter, cfg.maxVisibleClusters);
    b->visibleClusterCounter = counter;
    b->dispatchClassify = tc_dispatch_indirect{counter, 1, 1};
  } else if (mode == TC_BUILD_SETUP_DRAW_TESS) {
    uint32_t full = b->fullClusterCounter, part = b->partTriangleCounter;
    rb->numFullClusters = full;
    rb->numPartTriangles = part;
    rb->numSplitTriangles = b->splitWriteCounter;
    full = min(full, cfg.maxVisibleClusters);
    part = min(part, cfg.maxPartTriangles);
    b->drawFullClusters = tc_draw_mesh_tasks_indirect{full, 0};
    b->drawPartTriangles = tc_draw_mesh_tasks_indirect{(part + 31) / 32, 0};
    rb->numBlasClusters = full;
  } else if (mode == TC_BUILD_SETUP_SPLIT) {
    uint32_t count = min((uint32_t)b->splitTriangleCounter, cfg.maxSplitTriangles);
    b->splitWriteCounter = count;
    b->splitTriangleCounter = (int32_t)count;
    b->splitPassStart = 0;
    b->splitPassEnd = count;
    b->dispatchTriangleSplit = tc_dispatch_indirect{(count + 63) / 64, 1, 1};
  } else if (mode == TC_BUILD_SETUP_SPLIT_PASS) {
    b->splitPass = b->splitPass + 1;
    uint32_t start = min(b->splitPassEnd, cfg.maxSplitTriangles);
    uint32_t end = min(b->splitWriteCounter, cfg.maxSplitTriangles);
    b->splitPassStart = start;
    b->splitPassEnd = end;
    b->dispatchTriangleSplit = tc_dispatch_indirect{(end - start + 63) / 64, 1, 1};
  } else if (mode == TC_BUILD_SETUP_BUILD_BLAS) {
    const bool trans = transient_builds(cfg.flags);
    uint32_t temp = b->tempInstantiateCounter;
    uint32_t tr = trans ? b->transBuildCounter : 0u;
    rb->numBlasClusters = temp + tr;
    if (trans) rb->numTransBuilds = tr;
    rb->numTempInstantiations = temp;
    rb->numGenDatas = b->genClusterDataCounter;
    rb->numGenVertices = b->genVertexCounter;
    rb->numBlasReservedSizes = b->numBlasReservedSizes;
    temp = min(cfg.maxGeneratedClusters, temp);
    b->tempInstantiateCounter = temp;
    rb->numActualTempInstantiations = temp;
    b->dispatchBlasTempInsert = tc_dispatch_indirect{(temp + 63) / 64, 1, 1};
    if (trans) {
      tr = min(cfg.maxGeneratedClusters, temp + tr) - temp;
      b->transBuildCounter = tr;
      rb->numActualTransBuilds = tr;
      b->dispatchBlasTransInsert = tc_dispatch_indirect{(tr + 63) / 64, 1, 1};
    }
  } else if (mode == TC_BUILD_SETUP_INSTANTIATE_TESS) {
    const uint32_t part = b->partTriangleCounter;
    rb->numSplitTriangles = b->splitWriteCounter;
    if (transient_builds(cfg.flags)) {
      const uint32_t y = (uint32_t)(b->dualPartTriangleCounter >> 32);
      rb->numPartTriangles = part + y;
      rb->numTransPartTriangles = y;
    } else {
      rb->numPartTriangles = part;
    }
    const uint32_t ok = accepted_parts(a);
    b->partTriangleCounter = ok;
    b->dispatchTriangleInstantiate = tc_dispatch_indirect{(ok + 31) / 32, 1, 1};
  }
}

// The split's setups of the frame sequence, once its passes are done:
// SceneBuilding's split state as build_setup SPLIT and the SPLIT_PASSes leave
// it.  One thread.
__device__ __forceinline__ void split_state_one(const KArgs& a, uint32_t numPasses) {
  tc_scene_building* b = a.build;
  const SplitQueue* q = split_queue(a.ws);
  const SplitPass first = q->pass[0], last = q->pass[numPasses - 1];
  b->splitTriangleCounter = (int32_t)first.itemEnd;
  b->splitPass = b->splitPass + numPasses - 1;
  b->splitPassStart = last.itemBegin;
  b->splitPassEnd = last.itemEnd;
  b->dispatchTriangleSplit = tc_dispatch_indirect{(last.itemEnd - last.itemBegin + 63) / 64, 1, 1};
}

}  // namespace tc
