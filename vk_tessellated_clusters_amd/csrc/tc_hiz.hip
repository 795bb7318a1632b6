// tc_hiz.hip -- the far HiZ pyramid of a depth image (nvhiz_vk.cpp:278-320,
// nvhiz-update.comp.glsl with hizFarLevel 0 and standard depth): level 0
// holds the maximum of each 2 x 2 block of the depth image, every further
// level the maximum of 2 x 2 texels of the level before.  A launch makes six
// levels; reads of the source image clamp to its last row / column, so the
// whole power-of-two allocation is defined.
#include <algorithm>

#include "tc_kernels.h"

namespace tc {

__global__ void k_hiz_fill(float* t, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    t[i] = 1.0f;
}

// A workgroup makes the texels over 32 x 32 texels of level `first` in
// kHizLevels levels: first .. first + 5, each from the one before in LDS.
// What bounds a pyramid is its launches, not its bytes: with one launch per
// level a 1600 x 900 image took 61 us, 46 of them in ten launches over levels
// that together are a third of level 0's size.  Two launches take 16 + 5 us; the
// first one reads a float of every 48-byte record, 69 MB of lines at 4.3 TB/s.
constexpr uint32_t kHizTile = 32, kHizLevels = 6;

__device__ __forceinline__ float max2x2(float a, float b, float c, float d) { return fmaxf(fmaxf(fmaxf(a, b), c), d); }

// `at(px, py)`: the source of level `first`, the image or the level before.
template <typename Source>
__device__ __forceinline__ void hiz_tile(const tc_hiz& h, uint32_t first, Source at) {
  __shared__ float s_tile[2][kHizTile][kHizTile + 1];
  const uint32_t tx = blockIdx.x * kHizTile, ty = blockIdx.y * kHizTile;
  uint32_t dim = h.size >> first;
  float* dst = h.texels + hiz_level_offset(h.size, first);
  const uint32_t lx = threadIdx.x % kHizTile, ly = threadIdx.x / kHizTile;
  float m[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    // (past the last texel of a level smaller than the tile: that texel)
    const uint32_t x = min(tx + lx, dim - 1), y = min(ty + ly + 8 * i, dim - 1);
    m[i] = max2x2(at(2 * x, 2 * y), at(2 * x + 1, 2 * y), at(2 * x, 2 * y + 1), at(2 * x + 1, 2 * y + 1));
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t x = tx + lx, y = ty + ly + 8 * i;
    if (x < dim && y < dim) dst[(uint64_t)y * dim + x] = m[i];
    s_tile[0][ly + 8 * i][lx] = m[i];
  }
#pragma unroll
  for (uint32_t k = 1; k < kHizLevels; k++) {
    if (first + k >= h.mipLevels) break;
    dst += (uint64_t)dim * dim;
    dim >>= 1;
    __syncthreads();
    const uint32_t side = kHizTile >> k;
    if (threadIdx.x < side * side) {
      const uint32_t x = threadIdx.x % side, y = threadIdx.x / side;
      const auto& src = s_tile[(k - 1) & 1];
      const float v = max2x2(src[2 * y][2 * x], src[2 * y][2 * x + 1], src[2 * y + 1][2 * x], src[2 * y + 1][2 * x + 1]);
      s_tile[k & 1][y][x] = v;
      const uint32_t gx = (tx >> k) + x, gy = (ty >> k) + y;
      if (gx < dim && gy < dim) dst[(uint64_t)gy * dim + gx] = v;
    }
  }
}

__global__ __launch_bounds__(256) void k_hiz_image(tc_hiz h, const char* depth, uint32_t stride) {
  hiz_tile(h, 0, [&](uint32_t px, uint32_t py) {
    return *reinterpret_cast<const float*>(
        depth + ((uint64_t)min(py, h.height - 1) * h.width + min(px, h.width - 1)) * stride);
  });
}

__global__ __launch_bounds__(256) void k_hiz_down(tc_hiz h, uint32_t first) {
  const float* src = h.texels + hiz_level_offset(h.size, first - 1);
  const uint64_t dim = h.size >> (first - 1);
  hiz_tile(h, first, [&](uint32_t px, uint32_t py) { return src[py * dim + px]; });
}

static bool hiz_ok(const tc_hiz* h) {
  return h && h->texels && h->size && !(h->size & (h->size - 1)) && h->mipLevels >= 1 && h->mipLevels <= 16 &&
         (h->size >> (h->mipLevels - 1)) == 1 && h->width && h->height;
}

}  // namespace tc

using namespace tc;

extern "C" {

tc_status tc_hiz_setup(uint32_t width, uint32_t height, tc_hiz* hiz, uint64_t* bytes, float sizeFactors[4],
                       float* sizeMax) {
  // at least 3 used texels per axis, so the clamp factors (used - 2) stay
  // positive
  if (!hiz || width < 6 || height < 6 || width > (1u << 16) || height > (1u << 16)) return TC_ERROR_INVALID_ARGUMENT;
  // nvhiz_vk.cpp:290-310 with divisor 2 << hizFarLevel = 2
  const uint32_t dim = std::max(width, height) / 2;
  uint32_t size = 1, mips = 1;
  while (size < dim) size *= 2, mips++;
  hiz->size = size;
  hiz->mipLevels = mips;
  hiz->usedWidth = width / 2;
  hiz->usedHeight = height / 2;
  hiz->width = width;
  hiz->height = height;
  uint64_t n = 0;
  for (uint32_t k = 0; k < mips; k++) n += (uint64_t)(size >> k) * (size >> k);
  if (bytes) *bytes = 4 * n;
  // nvhiz_vk.cpp:29-40 getShaderFactors / getSizeMax
  if (sizeFactors) {
    sizeFactors[0] = float(hiz->usedWidth) / float(size);
    sizeFactors[1] = float(hiz->usedHeight) / float(size);
    sizeFactors[2] = float(hiz->usedWidth - 2) / float(size);
    sizeFactors[3] = float(hiz->usedHeight - 2) / float(size);
  }
  if (sizeMax) *sizeMax = float(size);
  return TC_OK;
}

tc_status tc_hiz_clear(const tc_hiz* hiz, tc_stream stream) {
  if (!hiz_ok(hiz)) return TC_ERROR_INVALID_ARGUMENT;
  uint64_t n = 0;
  for (uint32_t k = 0; k < hiz->mipLevels; k++) n += (uint64_t)(hiz->size >> k) * (hiz->size >> k);
  hipLaunchKernelGGL(k_hiz_fill, dim3((uint32_t)std::min<uint64_t>((n + 255) / 256, 4096)), dim3(256), 0, (hipStream_t)stream,
                     hiz->texels, n);
  return hipGetLastError() == hipSuccess ? TC_OK : TC_ERROR_LAUNCH;
}

tc_status tc_hiz_build(const tc_hiz* hiz, const void* depth, uint32_t pixelStride, tc_stream stream) {
  if (!hiz_ok(hiz) || !depth || pixelStride < 4 || (pixelStride & 3) || (reinterpret_cast<uintptr_t>(depth) & 3))
    return TC_ERROR_INVALID_ARGUMENT;
  hipStream_t st = (hipStream_t)stream;
  const tc_hiz h = *hiz;
  for (uint32_t k = 0; k < h.mipLevels; k += kHizLevels) {
    const uint32_t tiles = ((h.size >> k) + kHizTile - 1) / kHizTile;
    if (k == 0)
      hipLaunchKernelGGL(k_hiz_image, dim3(tiles, tiles), dim3(256), 0, st, h, (const char*)depth, pixelStride);
    else
      hipLaunchKernelGGL(k_hiz_down, dim3(tiles, tiles), dim3(256), 0, st, h, k);
  }
  return hipGetLastError() == hipSuccess ? TC_OK : TC_ERROR_LAUNCH;
}

}  // extern "C"
