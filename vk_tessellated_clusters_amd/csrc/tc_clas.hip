// tc_clas.hip -- cluster acceleration structure (CLAS) instantiation.
//
// Replaces vkCmdBuildClusterAccelerationStructureIndirectNV in template
// instantiation mode (renderer_raytrace_clusters_tess.cpp:595-623): every
// TemplateInstantiateInfo names a template (triangle order of a pattern or
// a base cluster) and a vertex range; the result at tempClusterAddresses[i]
// is a self-contained block
//   tc_clas_header | group boxes | triangle words | vertices
// and tempClusterSizes[i] receives its size.  Transient build records
// (ClasBuildInfo, 1X clusters) produce the same block format.
#include <stddef.h>

#include <algorithm>

#include "tc_kernels.h"
#include "tc_bvh.h"
#include "tc_insert.h"

namespace tc {

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) v = fminf(v, __shfl_xor(v, d, kWave));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) v = fmaxf(v, __shfl_xor(v, d, kWave));
  return v;
}

__host__ __device__ __forceinline__ uint32_t r16(uint32_t v) { return (v + 15u) & ~15u; }

// Group boxes and header of a block whose triangle words (s_t) and
// vertices (s_v) are in LDS and already copied to the block; returns the
// block size and the block's box.  One wave.
__device__ __forceinline__ uint32_t finish_block(char* dst, const float* s_v, const uint32_t* s_t, uint32_t nt, uint32_t nv,
                                                 uint32_t clusterID, uint32_t vertexBase, float lo[3], float hi[3]) {
  const uint32_t lane = lane_id();
  const uint32_t ng = (nt + TC_CLAS_GROUP_TRIANGLES - 1) / TC_CLAS_GROUP_TRIANGLES;
  tc_aabb* groups = reinterpret_cast<tc_aabb*>(dst + sizeof(tc_clas_header));
  for (int c = 0; c < 3; c++) lo[c] = INFINITY, hi[c] = -INFINITY;
  for (uint32_t g = lane; g < ng; g += kWave) {
    float glo[3] = {INFINITY, INFINITY, INFINITY}, ghi[3] = {-INFINITY, -INFINITY, -INFINITY};
    const uint32_t t1 = min(nt, (g + 1) * TC_CLAS_GROUP_TRIANGLES);
    for (uint32_t t = g * TC_CLAS_GROUP_TRIANGLES; t < t1; t++) {
      const uint32_t w = s_t[t];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const uint32_t vi = (w >> (8 * k)) & 0xFF;
#pragma unroll
        for (int c = 0; c < 3; c++) {
          glo[c] = fminf(glo[c], s_v[vi * 3 + c]);
          ghi[c] = fmaxf(ghi[c], s_v[vi * 3 + c]);
        }
      }
    }
    tc_aabb box;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      box.lo[c] = glo[c];
      box.hi[c] = ghi[c];
      lo[c] = fminf(lo[c], glo[c]);
      hi[c] = fmaxf(hi[c], ghi[c]);
    }
    gst_record(groups + g, box);
  }
#pragma unroll
  for (int c = 0; c < 3; c++) {
    lo[c] = wave_min(lo[c]);
    hi[c] = wave_max(hi[c]);
  }
  // zero the 16-byte padding after each part so blocks are deterministic
  {
    const uint32_t g0 = (uint32_t)sizeof(tc_clas_header) + ng * 24u, g1 = (uint32_t)sizeof(tc_clas_header) + r16(ng * 24u);
    const uint32_t t0 = g1 + nt * 4u, t1 = g1 + r16(nt * 4u);
    const uint32_t v0 = t1 + nv * 12u, v1 = t1 + r16(nv * 12u);
    uint32_t* w = reinterpret_cast<uint32_t*>(dst);
    const uint32_t npad = (g1 - g0) / 4 + (t1 - t0) / 4 + (v1 - v0) / 4;
    for (uint32_t k = lane; k < npad; k += kWave) {
      const uint32_t a = (g1 - g0) / 4, b = a + (t1 - t0) / 4;
      const uint32_t byte = k < a ? g0 + 4 * k : (k < b ? t0 + 4 * (k - a) : v0 + 4 * (k - b));
      gst(w + byte / 4, 0u);
    }
  }
  if (lane == 0) {
    tc_clas_header h;
    h.lo[0] = lo[0], h.lo[1] = lo[1], h.lo[2] = lo[2];
    h.hi[0] = hi[0], h.hi[1] = hi[1], h.hi[2] = hi[2];
    h.clusterID = clusterID;
    h.counts = nt | (nv << 8) | (ng << 16);
    h.vertexBase = vertexBase;
    h._pad[0] = h._pad[1] = h._pad[2] = 0;
    gst_record(reinterpret_cast<tc_clas_header*>(dst), h);
  }
  return (uint32_t)sizeof(tc_clas_header) + r16(ng * 24u) + r16(nt * 4u) + r16(nv * 12u);
}

__device__ __forceinline__ uint32_t vertex_base(const tc_scene_building* b, uint64_t vbuf) {
  return vbuf >= b->genVertices ? (uint32_t)((vbuf - b->genVertices) / 12u) : 0xFFFFFFFFu;
}

// Sum over the lanes of this lane's row of 16 up to it (all lanes active).
__device__ __forceinline__ uint32_t row_scan(uint32_t v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);  // row_shr:8
  return v;
}

// Value of the lane whose index differs in bit 0 / bit 1 (within four lanes).
template <int CTRL>
__device__ __forceinline__ float quad_swap(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
constexpr int kSwap1 = 0xB1, kSwap2 = 0x4E;  // quad_perm [1,0,3,2], [2,3,0,1]

// A wave builds a run of up to kBatch records in rounds.  A round takes as
// many of them as fit its LDS (whole clusters of 81 vertices: three;
// tessellated parts of a few triangles: about 14) and works flat over their
// vertices, triangle words and groups, 64 at a time.  With 16 lanes to a
// record the launch was bound by its instructions and their waits, not by
// memory: a part of 7 triangles left most lanes idle in unrolled copies sized
// for 128 triangles.  The blocks are put together in LDS and leave in 16-byte
// stores, 1 KB a step: written piece by piece, the stores took 550 of 791 us
// at the 3840 x 2160 patch field (1.6 GB of blocks).  Measured: patch field
// 1218 -> 610 us (3.9 TB/s), 500 meshes 139 -> 107 us, grid64 112 -> 73 us, 8192
// parts of 75 triangles 10 -> 9.2 us.  VALU is then 57 % busy.  Prefetching the
// next run's records gained 5 % at the patch field and lost as much at grid64;
// five waves per SIMD instead of four measured no difference.
constexpr uint32_t kBatch = 16;
constexpr uint32_t kRoundVerts = 256;  // at least kMaxClusterVerts
constexpr uint32_t kRoundTris = 384;
constexpr uint32_t kRoundGroups = 128;
constexpr uint32_t kRoundBytes = 7168;      // blocks of the round
constexpr uint32_t kMaxTemplateTris = 256;  // tc_cluster_template_order's limit
constexpr uint32_t kClasWaves = 4;
constexpr uint32_t kClasResident = 16;  // waves of a CU that a short frame's records are dealt over
static_assert(kRoundVerts >= kMaxClusterVerts && kRoundTris >= kMaxTemplateTris &&
                  kRoundGroups >= kMaxTemplateTris / TC_CLAS_GROUP_TRIANGLES &&
                  kRoundBytes >= sizeof(tc_clas_header) + kMaxTemplateTris * 10 + kMaxClusterVerts * 12 + 48,
              "a record fits a round");

struct ClasWave {
  // the round's blocks as they go to memory, one after another; in words and
  // in the 16-byte chunks they are written by
  union {
    uint32_t u[kRoundBytes / 4];
    float f[kRoundBytes / 4];
    uint4 chunk[kRoundBytes / 16];
  };
  // the round's records, one 16-byte read per kind of item.  Addresses and
  // offsets are those that item 0 of the round would have if the record began
  // with it (modulo 2^64 and 2^16), so item i lies at base + i * its size.
  uint4 vert[kBatch];   // source address, stride, word offset of the vertices
  uint4 tri[kBatch];    // template words' address, word offset of the triangles
  uint4 group[kBatch];  // first group | triangles << 16, word offsets: triangles | vertices << 16, boxes,
                        // groups | vertices << 16
  uint4 block[kBatch];  // block address, cluster ID, counts
  uint2 head[kBatch];   // vertexBase, first chunk | chunks << 16
  // a bit for every first item of a record: vertices, triangles, groups, chunks
  uint64_t heads[kRoundVerts / 64 + kRoundTris / 64 + kRoundGroups / 64 + kRoundBytes / 16 / 64];
};
constexpr uint32_t kHeadT = kRoundVerts / 64, kHeadG = kHeadT + kRoundTris / 64, kHeadC = kHeadG + kRoundGroups / 64,
                   kHeads = kHeadC + kRoundBytes / 16 / 64;

__device__ __forceinline__ void mark_head(uint64_t* heads, uint32_t first) {
  __hip_atomic_fetch_or(reinterpret_cast<uint32_t*>(heads) + (first >> 5), 1u << (first & 31), __ATOMIC_RELAXED,
                        __HIP_MEMORY_SCOPE_WAVEFRONT);
}

__device__ __forceinline__ uint64_t u64(uint32_t lo, uint32_t hi) { return ((uint64_t)hi << 32) | lo; }

// Runs of records, grid-stride over tempInstantiateCounter; a frame with
// fewer than kBatch records for each of the chip's resident waves takes
// shorter runs (8192 records in runs of 1 on 40 waves a CU: 14 us, of 2 on 16
// waves: 9.5 us).  With an insertion plan, one workgroup more makes its setup
// and every record's Morton code is left for its keys.
__global__ __launch_bounds__(kClasWaves * kWave) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_clas_instantiate(KArgs a, uint32_t residentWaves, InsertPlan ip) {
  __shared__ ClasWave s_wave[kClasWaves];
  if (ip.state && blockIdx.x == 0) {
    static_assert(kClasWaves * kWave == kSortThreads && sizeof(s_wave) >= 4 * kInsertSetupWords, "setup workgroup");
    insert_setup(a, ip, reinterpret_cast<uint32_t*>(s_wave));
    return;
  }
  const uint32_t group = blockIdx.x - (ip.state ? 1 : 0), groups = gridDim.x - (ip.state ? 1 : 0);
  const tc_scene_building* b = a.build;
  const uint32_t n = min(b->tempInstantiateCounter, a.cfg.maxGeneratedClusters);
  const uint32_t lane = lane_id();
  ClasWave& w = s_wave[threadIdx.x / kWave];
  const tc_template_instantiate_info* infos = ptr<const tc_template_instantiate_info>(b->tempInstantiations);
  const uint64_t* dsts = ptr<const uint64_t>(b->tempClusterAddresses);
  const uint32_t* instances = ptr<const uint32_t>(b->tempInstanceIDs);
  uint32_t* sizes = ptr<uint32_t>(b->tempClusterSizes);
  const uint32_t waves = groups * kClasWaves;
  const uint32_t run = min(kBatch, max(1u, (n + residentWaves - 1) / residentWaves));
  for (uint32_t r0 = uniform(group * kClasWaves + threadIdx.x / kWave) * run; r0 < n; r0 += waves * run) {
    const uint32_t cnt = min(run, n - r0);
    // lanes 0 .. cnt - 1 hold the run's records
    const bool held = lane < cnt;
    uint64_t dst = 0, src = 0, words = 0;
    uint32_t stride = 12, nv = 0, nt = 0, clusterID = 0;
    float geo[6], box[6];  // of the lane's record: instance bounds, CLAS
    if (held) {
      const tc_template_instantiate_info info = gld_record(infos + r0 + lane);
      dst = gld(dsts + r0 + lane);
      const tc_clas_template T = gld_record(ptr<const tc_clas_template>(info.clusterTemplateAddress));
      src = info.vertexBufferAddress;
      stride = (uint32_t)info.vertexBufferStride;
      words = T.triangles;
      nv = min(T.numVertices, kMaxClusterVerts);
      nt = min(T.numTriangles, kMaxTemplateTris);
      clusterID = T.clusterID + info.clusterIdOffset;
      if (ip.state) {
        const tc_render_instance& ri = a.instances[gld(instances + r0 + lane)];
#pragma unroll
        for (int x = 0; x < 3; x++) geo[x] = gld(ri.geoLo + x), geo[3 + x] = gld(ri.geoHi + x);
      }
    }
    const uint32_t ng = (nt + TC_CLAS_GROUP_TRIANGLES - 1) / TC_CLAS_GROUP_TRIANGLES;
    const uint32_t oT = (uint32_t)sizeof(tc_clas_header) + r16(ng * 24u), oV = oT + r16(nt * 4u), size = oV + r16(nv * 12u);
    // a record without vertices or triangles takes a round of its own, so
    // that a round's first items are its records
    const bool empty = ballot(held && (nv == 0 || nt == 0)) != 0;
    for (uint32_t done = 0; done < cnt;) {
      // the records of this round: done .. done + k - 1
      const bool left = held && lane >= done && !(empty && lane > done);
      const uint32_t ev = row_scan(left ? nv : 0u), et = row_scan(left ? nt : 0u), eg = row_scan(left ? ng : 0u),
                     es = row_scan(left ? size : 0u);
      const uint64_t fit = ballot(left && ev <= kRoundVerts && et <= kRoundTris && eg <= kRoundGroups && es <= kRoundBytes);
      const uint32_t k = __popcll(fit), lastLane = done + k - 1;
      const uint32_t numV = __builtin_amdgcn_readlane(ev, lastLane), numT = __builtin_amdgcn_readlane(et, lastLane),
                     numG = __builtin_amdgcn_readlane(eg, lastLane), numC = __builtin_amdgcn_readlane(es, lastLane) / 16;
      const bool in = left && lane < done + k;
      if (lane < kHeads) w.heads[lane] = 0;
      wave_sync();
      if (in) {
        const uint32_t fv = ev - nv, ft = et - nt, fg = eg - ng, fs = es - size;
        const uint64_t sa = src - (uint64_t)fv * stride, wa = words - 4ull * ft, da = dst - fs;
        const uint32_t bT = (fs + oT) / 4, bV = (fs + oV) / 4, bG = (fs + (uint32_t)sizeof(tc_clas_header)) / 4;
        w.vert[lane] = make_uint4((uint32_t)sa, (uint32_t)(sa >> 32), stride, bV - 3 * fv);
        w.tri[lane] = make_uint4((uint32_t)wa, (uint32_t)(wa >> 32), bT - ft, 0u);
        w.group[lane] = make_uint4(fg | nt << 16, bT | bV << 16, bG, ng | nv << 16);
        w.block[lane] = make_uint4((uint32_t)da, (uint32_t)(da >> 32), clusterID, nt | (nv << 8) | (ng << 16));
        w.head[lane] = make_uint2(vertex_base(b, src), fs / 16 | (size / 16) << 16);
        mark_head(w.heads, fv);
        mark_head(w.heads + kHeadT, ft);
        mark_head(w.heads + kHeadG, fg);
        mark_head(w.heads + kHeadC, fs / 16);
      }
      wave_sync();
      // word j of the heads in lane j; the record of item 64 * j + lane of a
      // kind, `before` counting the first items in earlier words
      const uint64_t headWord = lane < kHeads ? w.heads[lane] : 0ull;
      auto record = [&](uint32_t word, uint32_t& before) {
        const uint64_t h = u64(__builtin_amdgcn_readlane((uint32_t)headWord, word),
                               __builtin_amdgcn_readlane((uint32_t)(headWord >> 32), word));
        const uint32_t q = before + (uint32_t)(h & 1) + mask_prefix(h >> 1) - 1;
        before += __popcll(h);
        return q & (kBatch - 1);
      };
      // vertices and triangle words: every load of the round, then the image.
      // Lanes past the end repeat the last item, so that no branch lies
      // between the loads (one would make a load wait for the one before).
      if (numV != 0 && numT != 0) {
        float vx[kRoundVerts / 64][3];
        uint32_t tw[kRoundTris / 64], va[kRoundVerts / 64], ta[kRoundTris / 64];
        uint32_t before = done;
#pragma unroll
        for (uint32_t j = 0; j < kRoundVerts / 64; j++) {
          const uint4 r = w.vert[record(j, before)];
          const uint32_t i = min(64 * j + lane, numV - 1);
          const gfloat3 f = gld3(ptr<const float>(u64(r.x, r.y) + (uint64_t)i * r.z));
          vx[j][0] = f.x, vx[j][1] = f.y, vx[j][2] = f.z;
          va[j] = r.w + 3 * i;
        }
        before = done;
#pragma unroll
        for (uint32_t j = 0; j < kRoundTris / 64; j++) {
          const uint4 r = w.tri[record(kHeadT + j, before)];
          const uint32_t i = min(64 * j + lane, numT - 1);
          tw[j] = gld(ptr<const uint32_t>(u64(r.x, r.y)) + i);
          ta[j] = r.z + i;
        }
#pragma unroll
        for (uint32_t j = 0; j < kRoundVerts / 64; j++)
          w.f[va[j]] = vx[j][0], w.f[va[j] + 1] = vx[j][1], w.f[va[j] + 2] = vx[j][2];
#pragma unroll
        for (uint32_t j = 0; j < kRoundTris / 64; j++) w.u[ta[j]] = tw[j];
      } else {
        // a record of vertices or of triangles alone, in its own round
        const uint4 rv = w.vert[done], rt = w.tri[done];
        for (uint32_t i = lane; i < numV; i += kWave) {
          const gfloat3 f = gld3(ptr<const float>(u64(rv.x, rv.y) + (uint64_t)i * rv.z));
          float* v = w.f + rv.w + 3 * i;
          v[0] = f.x, v[1] = f.y, v[2] = f.z;
        }
        for (uint32_t i = lane; i < numT; i += kWave) w.u[rt.z + i] = gld(ptr<const uint32_t>(u64(rt.x, rt.y)) + i);
      }
      wave_sync();
      // group boxes
      {
        uint32_t before = done;
#pragma unroll
        for (uint32_t j = 0; j < kRoundGroups / 64; j++) {
          if (64 * j >= numG) continue;
          const uint32_t i = 64 * j + lane, q = record(kHeadG + j, before);
          if (i < numG) {
            const uint4 r = w.group[q];
            const uint32_t g = i - (r.x & 0xFFFF), t0 = g * TC_CLAS_GROUP_TRIANGLES, rnt = r.x >> 16;
            const uint4 w4 = *reinterpret_cast<const uint4*>(w.u + (r.y & 0xFFFF) + t0);
            // past the last triangle the one before again
            uint32_t word[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
            for (uint32_t m = 1; m < TC_CLAS_GROUP_TRIANGLES; m++) word[m] = t0 + m < rnt ? word[m] : word[m - 1];
            const float* v = w.f + (r.y >> 16);
            float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
#pragma unroll
            for (uint32_t m = 0; m < TC_CLAS_GROUP_TRIANGLES; m++) {
#pragma unroll
              for (int c = 0; c < 3; c++) {
                const float* p = v + 3 * ((word[m] >> (8 * c)) & 0xFF);
#pragma unroll
                for (int x = 0; x < 3; x++) lo[x] = fminf(lo[x], p[x]), hi[x] = fmaxf(hi[x], p[x]);
              }
            }
            float* box = w.f + r.z + 6 * g;
#pragma unroll
            for (int x = 0; x < 3; x++) box[x] = lo[x], box[3 + x] = hi[x];
          }
        }
      }
      wave_sync();
      // headers, four lanes to a record, and the zeros after each part
      {
        const uint32_t q = lane >> 2, sl = lane & 3;
        const bool mine = q >= done && q < done + k;
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        const uint4 r = w.group[q];
        const uint32_t rng = mine ? r.w & 0xFFFF : 0u;
        for (uint32_t g = sl; g < rng; g += 4) {
          const float* bx = w.f + r.z + 6 * g;
#pragma unroll
          for (int x = 0; x < 3; x++) lo[x] = fminf(lo[x], bx[x]), hi[x] = fmaxf(hi[x], bx[3 + x]);
        }
#pragma unroll
        for (int x = 0; x < 3; x++) {
          lo[x] = fminf(lo[x], quad_swap<kSwap1>(lo[x])), hi[x] = fmaxf(hi[x], quad_swap<kSwap1>(hi[x]));
          lo[x] = fminf(lo[x], quad_swap<kSwap2>(lo[x])), hi[x] = fmaxf(hi[x], quad_swap<kSwap2>(hi[x]));
        }
        if (mine) {
          const uint4 bl = w.block[q];
          const uint2 hd = w.head[q];
          const uint32_t bT = r.y & 0xFFFF, bV = r.y >> 16, rnv = r.w >> 16;
          const uint32_t g0 = r.z + 6 * rng + sl, t0 = bT + (r.x >> 16) + sl, end = ((hd.y & 0xFFFF) + (hd.y >> 16)) * 4;
          if (g0 < bT) w.u[g0] = 0;
          if (t0 < bV) w.u[t0] = 0;
          if (bV + 3 * rnv + sl < end) w.u[bV + 3 * rnv + sl] = 0;
          uint4 h = make_uint4(hd.x, 0u, 0u, 0u);
          if (sl == 0) h = make_uint4(__float_as_uint(lo[0]), __float_as_uint(lo[1]), __float_as_uint(lo[2]), bl.z);
          if (sl == 1) h = make_uint4(__float_as_uint(hi[0]), __float_as_uint(hi[1]), __float_as_uint(hi[2]), bl.w);
          if (sl < 3) w.chunk[(hd.y & 0xFFFF) + sl] = h;
        }
      }
      static_assert(sizeof(tc_clas_header) == 48 && offsetof(tc_clas_header, clusterID) == 12 &&
                        offsetof(tc_clas_header, counts) == 28 && offsetof(tc_clas_header, vertexBase) == 32,
                    "the header as three chunks");
      wave_sync();
      // the image to memory, 1 KB a step
      if (in) {
        gst(sizes + r0 + lane, size);
        if (ip.state) {
          const float* h = w.f + 4 * (w.head[lane].y & 0xFFFF);
#pragma unroll
          for (int x = 0; x < 3; x++) box[x] = h[x], box[3 + x] = h[4 + x];
        }
      }
      {
        uint32_t before = done;
#pragma unroll
        for (uint32_t j = 0; j < kRoundBytes / 16 / 64; j++) {
          if (64 * j >= numC) continue;
          const uint32_t i = 64 * j + lane, q = record(kHeadC + j, before);
          if (i < numC) {
            const uint4 c = w.chunk[i];
            const uint2 d = *reinterpret_cast<const uint2*>(&w.block[q]);
            typedef uint32_t u4 __attribute__((ext_vector_type(4), aligned(4)));
            gst(ptr<u4>(u64(d.x, d.y)) + i, u4{c.x, c.y, c.z, c.w});
          }
        }
      }
      wave_sync();
      done += k;
    }
    if (ip.state && held) gst(ip.codes + r0 + lane, morton24_of(box, box + 3, geo, geo + 3));
  }
}

constexpr uint32_t kWaveFloatsPerLane = (kMaxClusterVerts * 3 + kWave - 1) / kWave;
constexpr uint32_t kWaveTrisPerLane = (kMaxClusterTris + kWave - 1) / kWave;

// Transient builds (stands for the NV transient CLAS build,
// renderer_raytrace_clusters_tess.cpp:625-655): triangles in record order
// with the transient triangle index as primitive, all the record's
// vertices.  One wave per CLAS, grid-stride over transBuildCounter.  With
// `codes`, as k_clas_instantiate.
__global__ __launch_bounds__(64) void k_clas_build_transient(KArgs a, uint32_t* codes) {
  __shared__ float s_v[kMaxClusterVerts * 3];
  __shared__ uint32_t s_t[kMaxClusterTris];
  const tc_scene_building* b = a.build;
  const uint32_t n = min(b->transBuildCounter, a.cfg.maxGeneratedClusters);
  const uint32_t lane = lane_id();
  const tc_clas_build_info* infos = ptr<const tc_clas_build_info>(b->transBuilds);
  const uint64_t* dsts = ptr<const uint64_t>(b->transClusterAddresses);
  uint32_t* sizes = ptr<uint32_t>(b->transClusterSizes);
  for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
    const tc_clas_build_info info = gld_record(infos + i);
    const uint32_t nt = min(info.packed & 511u, kMaxClusterTris), nv = min((info.packed >> 9) & 511u, kMaxClusterVerts);
    const uint32_t ng = (nt + TC_CLAS_GROUP_TRIANGLES - 1) / TC_CLAS_GROUP_TRIANGLES;
    char* dst = ptr<char>(gld(dsts + i));
    uint32_t* tris = reinterpret_cast<uint32_t*>(dst + sizeof(tc_clas_header) + r16(ng * 24u));
    float* verts = reinterpret_cast<float*>(dst + sizeof(tc_clas_header) + r16(ng * 24u) + r16(nt * 4u));
    const char* src = ptr<const char>(info.vertexBuffer);
    const uint8_t* ix = ptr<const uint8_t>(info.indexBuffer);
    const uint32_t is = info.indexBufferStride;
    // the loads of a record are issued together (packed vertices from one
    // base), so the copy waits for one round trip rather than one per element
    const uint32_t nf = nv * 3;
    if (info.vertexBufferStride == 12u) {
      const float* vs = reinterpret_cast<const float*>(src) + lane;
      float vf[kWaveFloatsPerLane];
#pragma unroll
      for (uint32_t j = 0; j < kWaveFloatsPerLane; j++) vf[j] = lane + j * kWave < nf ? gld(vs + j * kWave) : 0.0f;
#pragma unroll
      for (uint32_t j = 0; j < kWaveFloatsPerLane; j++) {
        const uint32_t k = lane + j * kWave;
        if (k < nf) s_v[k] = vf[j], gst(verts + k, vf[j]);
      }
    } else {
      for (uint32_t k = lane; k < nf; k += kWave) {
        const uint32_t v = k / 3, c = k - v * 3;
        const float f = gld(reinterpret_cast<const float*>(src + (uint64_t)v * info.vertexBufferStride) + c);
        s_v[k] = f;
        gst(verts + k, f);
      }
    }
    uint32_t tb[kWaveTrisPerLane][3];
#pragma unroll
    for (uint32_t j = 0; j < kWaveTrisPerLane; j++) {
      const uint32_t t = lane + j * kWave;
      const uint8_t* q = ix + (uint64_t)(t < nt ? t : 0u) * 3u * is;
      tb[j][0] = t < nt ? (uint32_t)gld(q) : 0u;
      tb[j][1] = t < nt ? (uint32_t)gld(q + is) : 0u;
      tb[j][2] = t < nt ? (uint32_t)gld(q + 2u * is) : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < kWaveTrisPerLane; j++) {
      const uint32_t t = lane + j * kWave;
      if (t < nt) {
        const uint32_t w = tb[j][0] | (tb[j][1] << 8) | (tb[j][2] << 16) | (t << 24);
        s_t[t] = w;
        gst(tris + t, w);
      }
    }
    __syncthreads();
    float lo[3], hi[3];
    const uint32_t size = finish_block(dst, s_v, s_t, nt, nv, info.clusterID, vertex_base(b, info.vertexBuffer), lo, hi);
    if (lane == 0) gst(sizes + i, size);
    if (codes && lane == 0) {
      const tc_render_instance& ri = a.instances[gld(ptr<const uint32_t>(b->transInstanceIDs) + i)];
      const uint32_t numTemp = min(b->tempInstantiateCounter, a.cfg.maxGeneratedClusters);
      if (numTemp + i < a.cfg.maxGeneratedClusters) gst(codes + numTemp + i, morton24_of(lo, hi, ri.geoLo, ri.geoHi));
    }
    __syncthreads();
  }
}

}  // namespace tc

using namespace tc;

static tc_status launch_clas(const tc_bindings* b, tc_config config, tc_stream stream, const InsertPlan& ip) {
  KArgs a;
  tc_status s = make_args_public(b, config, a);
  if (s != TC_OK) return s;
  const uint32_t waves = std::min<uint32_t>((config.maxGeneratedClusters + 3) / 4,
                                            (uint32_t)num_cu_public() * tuning_snapshot().clasWavesPerCU);
  const uint32_t grid = (waves + kClasWaves - 1) / kClasWaves;
  hipLaunchKernelGGL(k_clas_instantiate, dim3(grid + (ip.state ? 1 : 0)), dim3(kClasWaves * kWave), 0, (hipStream_t)stream, a,
                     (uint32_t)num_cu_public() * kClasResident, ip);
  return hipGetLastError() == hipSuccess ? TC_OK : TC_ERROR_LAUNCH;
}

extern "C" tc_status tc_clas_instantiate(const tc_bindings* b, tc_config config, tc_stream stream) {
  return launch_clas(b, config, stream, InsertPlan{});
}

static tc_status launch_transient(const tc_bindings* b, tc_config config, tc_stream stream, uint32_t* codes) {
  KArgs a;
  tc_status s = make_args_public(b, config, a);
  if (s != TC_OK) return s;
  if (!transient_builds(config.flags)) return TC_OK;
  uint32_t grid = std::min<uint32_t>(config.maxGeneratedClusters, (uint32_t)num_cu_public() * tuning_snapshot().clasWavesPerCU);
  hipLaunchKernelGGL(k_clas_build_transient, dim3(grid), dim3(64), 0, (hipStream_t)stream, a, codes);
  return hipGetLastError() == hipSuccess ? TC_OK : TC_ERROR_LAUNCH;
}

extern "C" tc_status tc_clas_build_transient(const tc_bindings* b, tc_config config, tc_stream stream) {
  return launch_transient(b, config, stream, nullptr);
}

tc_status tc::clas_build_setup(const tc_bindings* b, tc_config config, tc_stream stream) {
  if (!b || !b->workspace) return TC_ERROR_INVALID_ARGUMENT;
  const InsertPlan ip = insert_plan(b, config);
  const tc_status s = launch_clas(b, config, stream, ip);
  return s != TC_OK ? s : launch_transient(b, config, stream, ip.codes);
}
