// tc_insert.h -- the renderer's BLAS insertion and key sort as one sort.
//
// blas_setup_insertion, the insertion and the BLAS key sort are 8 to 14 small
// launches when each stands for itself (one workgroup; upsweep, passes and
// scatter; keys, upsweep and passes), and a small launch between two others
// takes about 4.5 us whatever it does.  Where the three follow each other:
//   * one workgroup of the CLAS launch makes the setup, since the reference
//     counts are final before it, and with them the digit bases of every pass
//     over instance digits: the lists' starts are prefix sums of the counts;
//   * the CLAS launches leave each CLAS's Morton code with its block, from the
//     box they have at hand;
//   * the insertion's last pass writes each CLAS address and its BLAS key at
//     their final places and counts the keys' Morton digits, so neither the
//     scatter, the key launch (which read every header again) nor an upsweep is
//     left.
// Launches from the CLAS to the tree: one instance 10 -> 4, up to 256 instances
// 10 -> 5, more 13 -> 7.  Frames: icosphere at 320 x 180 260 -> 242 us, grid64 1012
// -> 986, 500 meshes 1610 -> 1582, patch field at 3840 x 2160 6747 -> 6550.
#pragma once

#include "tc_sort.h"

namespace tc {

constexpr uint32_t kMortonPasses = 3;

struct InsertPlan {
  SortState* state;  // null: no insertion follows
  uint64_t* status;
  uint32_t* codes;  // Morton codes, templates first (value slot 1, free until the key passes)
  uint32_t maxTiles;
  uint32_t capacity;
  uint32_t insertPasses;    // 1 for up to 256 instances, else 2
  uint32_t instancePasses;  // of the key sort: as many, none for one instance
};

// Rounds of kSortThreads CLAS in an insertion tile, n in all: halved from
// kSortKeysPerThread while that leaves fewer than kInsertTiles tiles (each has
// a row of status words).  26k CLAS: last pass 19 us with 16 tiles, 15 with 64
// or 128; 168k: 34, 34 and 28 us.  The key passes keep their full tiles: with
// little besides the walk to do, they are slower with more of them (125k keys:
// 12.3 us in 61 tiles, 15.6 in 122).
constexpr uint32_t kInsertTiles = 128;
__host__ __device__ __forceinline__ uint32_t insert_tiles(uint32_t n, uint32_t rounds) {
  return (n + rounds * kSortThreads - 1) / (rounds * kSortThreads);
}
__device__ __forceinline__ uint32_t insert_rounds(uint32_t n, uint32_t maxTiles) {
  uint32_t r = kSortKeysPerThread;
  while (r > 1 && insert_tiles(n, r) < kInsertTiles && insert_tiles(n, r / 2) <= maxTiles) r /= 2;
  return r;
}
// Tiles of up to `capacity` CLAS at any number of rounds, at most.
inline uint32_t insert_grid(uint32_t capacity, uint32_t maxTiles) {
  const uint32_t most = std::max(insert_tiles(capacity, kSortKeysPerThread), std::min(insert_tiles(capacity, 1), 2 * kInsertTiles));
  return std::max(1u, std::min(most, maxTiles));
}

InsertPlan insert_plan(const tc_bindings* b, const tc_config& config);
// The CLAS of both lists, with the insertion's setup and their Morton codes.
tc_status clas_build_setup(const tc_bindings* b, tc_config config, tc_stream stream);
// The insertion after it: reference lists, size total, and the keys and values
// of slot 0.
tc_status insert_clusters(const tc_bindings* b, tc_config config, tc_stream stream);
// tc_accel_build on the keys that insert_clusters left.
tc_status accel_build_inserted(const tc_bindings* b, tc_config config, const tc_accel* accel, const float* instanceXforms,
                               tc_stream stream);

// blas_setup_insertion (blas_setup_insertion.comp.glsl:100-116, the lists
// starting at the array's start) and the plan's sort state, by one workgroup
// of kSortThreads threads, four instances a thread.  The counts stay as they
// are: they are what the insertion will have inserted.
constexpr uint32_t kInsertSetupWords = kSortRadix + 8;
__device__ __forceinline__ void insert_setup(const KArgs& a, const InsertPlan& ip, uint32_t* lds /* kInsertSetupWords */) {
  uint32_t *s_hist = lds, *s_wave = lds + kSortRadix, *s_sizes = s_wave + 4;
  tc_scene_building* b = a.build;
  SortState* st = ip.state;
  tc_blas_build_info* infos = ptr<tc_blas_build_info>(b->blasBuildInfos);
  const uint32_t* sizes = ptr<const uint32_t>(b->blasBuildSizes);
  const uint64_t refs = b->blasClusterAddresses;
  const uint32_t t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  const uint32_t keyPass = ip.insertPasses + kMortonPasses;  // the key sort's instance digits
  const uint32_t passes = keyPass + ip.instancePasses;
  const uint32_t last = st->epoch, e0 = sort_epoch0(last, passes);
  if (e0 != last + 1)
    for (uint64_t i = t; i < (uint64_t)ip.maxTiles * kSortRadix; i += kSortThreads) ip.status[i] = 0;
  s_hist[t] = 0;
  if (t == 0) *s_sizes = 0;
  uint32_t carry = 0, sizeSum = 0;
  __syncthreads();
  for (uint32_t i0 = 0; i0 < a.numInstances; i0 += 4 * kSortThreads) {
    uint32_t cnt[4], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
      const uint32_t i = i0 + 4 * t + j;
      cnt[j] = i < a.numInstances ? infos[i].clusterReferencesCount : 0u;
      sizeSum += i < a.numInstances ? sizes[i] : 0u;
      sum += cnt[j];
    }
    const uint32_t incl = wave_incl_scan(sum);
    if (lane == kWave - 1) s_wave[wave] = incl;
    __syncthreads();
    uint32_t off = carry + incl - sum;
#pragma unroll
    for (uint32_t w = 0; w < kSortThreads / kWave; w++) {
      if (w < wave) off += s_wave[w];
      carry += s_wave[w];
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
      const uint32_t i = i0 + 4 * t + j;
      if (i < a.numInstances) {
        tc_blas_build_info bi;
        bi.clusterReferencesCount = cnt[j];
        bi.clusterReferencesStride = 8;
        bi.clusterReferences = refs + (uint64_t)off * 8ull;
        infos[i] = bi;
        // an instance digit's first position: the start of its instance, of
        // its first instance for the high digit
        if (ip.insertPasses == 1) {
          st->bases[0][i] = st->bases[keyPass][i] = off;
        } else {
          if (cnt[j]) atomicAdd(&s_hist[i & 255u], cnt[j]);
          if ((i & 255u) == 0) st->bases[1][i >> 8] = st->bases[keyPass + 1][i >> 8] = off;
        }
        off += cnt[j];
      }
    }
    __syncthreads();
  }
  sizeSum = wave_sum(sizeSum);
  if (lane == 0) atomicAdd(s_sizes, sizeSum);
  __syncthreads();
  if (ip.insertPasses > 1 && wave == 0) {  // the low digit's, over all instances
    uint32_t v[4], sum = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = s_hist[4 * lane + j], sum += v[j];
    uint32_t run = wave_incl_scan(sum) - sum;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      st->bases[0][4 * lane + j] = st->bases[keyPass][4 * lane + j] = run;
      run += v[j];
    }
  }
  if (t == 0) {
    b->blasClusterCounter = carry;
    a.readback->numBlasActualSizes += *s_sizes;
    for (uint32_t p = 0; p < kSortMaxPasses; p++) st->ticket[p] = 0;
    st->epoch0 = e0;
    st->epoch = e0 + passes - 1;
  }
}

}  // namespace tc
