// LDS staging of transient rows for the kernels that gather from all rows at
// every voxel, gfx950.
#pragma once

#include "common.h"

namespace totri_hip {
namespace {

// Staged rows (A2, A3, A5): two LDS buffers of `cap` floats.  A workgroup writes
// the next rows, loaded into registers one stage earlier, into one buffer
// while its waves read the other, so a stage costs one barrier.  Every
// workgroup reads all rows, so L2 traffic falls with the voxels per workgroup:
// at 64^3 and 4096 pairs of 512 bins, 1024 lanes (one workgroup per CU) read
// 2.1 GB where 256 lanes read 8.6 GB (A3: 0.85 -> 0.79 ms).  Volumes that
// would leave a quarter of the CUs without a workgroup of 1024 keep 256 lanes.
// Floats per buffer, at most: 72 KiB, where a workgroup has a CU to itself.
constexpr int kStageMax = 18432;

template <int NTH>
struct RowStage {
  static constexpr int kCopy4 = (kStageMax / 4 + NTH - 1) / NTH;
  float4 buf[kCopy4];
  // n4 float4s, 0 <= n4 <= kStageMax / 4
  __device__ __forceinline__ void load(const float* src, int n4) {
#pragma unroll
    for (int i = 0; i < kCopy4; ++i) {
      const int e = i * NTH + (int)threadIdx.x;
      buf[i] = e < n4 ? ((const float4*)src)[e] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  // The same from pieces of `piece` float4s that start `step` float4s apart.
  __device__ __forceinline__ void load_pieces(const float* src, int n4, int piece, int64_t step) {
#pragma unroll
    for (int i = 0; i < kCopy4; ++i) {
      const int e = i * NTH + (int)threadIdx.x;
      const int k = e / piece;
      buf[i] = e < n4 ? ((const float4*)src)[k * step + (e - k * piece)]
                      : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  __device__ __forceinline__ void store(float* dst, int n4) const {
#pragma unroll
    for (int i = 0; i < kCopy4; ++i) {
      const int e = i * NTH + (int)threadIdx.x;
      if (e < n4) ((float4*)dst)[e] = buf[i];
    }
  }
};

// Lets a kernel take both buffers (launches get 64 KiB by default).
template <typename K>
int allow_stage(K kernel) {
  TOTRI_CHECK_HIP(hipFuncSetAttribute((const void*)kernel,
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      2 * kStageMax * (int)sizeof(float)));
  return TOTRI_OK;
}

// Workgroup size and floats per buffer for B volumes of nvox voxels.
struct StagePlan {
  int threads, cap;
};

StagePlan stage_plan(int64_t B, int64_t nvox) {
  if (B * ((nvox + 1023) / 1024) >= 192) return {1024, kStageMax};
  // two buffers per workgroup of the CU's 160 KiB: one to four of them
  const int64_t blocks = B * ((nvox + 255) / 256);
  return {256, blocks <= 256 ? kStageMax : blocks <= 512 ? 10240 : blocks <= 768 ? 6720 : 5120};
}

}  // namespace
}  // namespace totri_hip
