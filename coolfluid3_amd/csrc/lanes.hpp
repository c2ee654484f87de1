// Cross-lane sums by DPP: register moves between the lanes of a row of 16, a few cycles each, where a
// shuffle goes through the LDS permute unit (two ds_bpermute per double and step, about 100 cycles).  On the
// small launches of the Krylov loop the reductions are most of what a wave waits for after its loads.
#pragma once

#include <hip/hip_runtime.h>

namespace cf3hip {
namespace lanes {

// the value of the lane that DPP control CTRL names (all lanes active)
template<int CTRL>
__device__ __forceinline__ float move(float x)
{
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template<int CTRL>
__device__ __forceinline__ double move(double x)
{
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

constexpr int kXor1 = 0xB1, kXor2 = 0x4E;          // quad_perm [1,0,3,2], [2,3,0,1]
constexpr int kHalfMirror = 0x141, kMirror = 0x140; // lane i <- 7 - i of its 8, 15 - i of its 16
constexpr int kNext4 = 0x12C, kNext8 = 0x128;       // lane i <- i + 4, i + 8 of its 16, around

// sum over each row of 16 lanes, in every lane of it; over each 8 lanes
template<typename T>
__device__ __forceinline__ T sum8(T x)
{
  x += move<kXor1>(x);
  x += move<kXor2>(x);
  x += move<kHalfMirror>(x);
  return x;
}
template<typename T>
__device__ __forceinline__ T sum16(T x)
{
  x = sum8(x);
  x += move<kMirror>(x);
  return x;
}

__device__ __forceinline__ double read_lane(double x, int lane)
{
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}

// sum over the 64 lanes, in every lane
__device__ __forceinline__ double sum64(double x)
{
  x = sum16(x);
  return (read_lane(x, 0) + read_lane(x, 16)) + (read_lane(x, 32) + read_lane(x, 48));
}

}  // namespace lanes
}  // namespace cf3hip
