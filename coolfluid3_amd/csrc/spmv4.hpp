// Row kernels of the neq = 4 block-CSR product (16 lanes per node row), shared by the plain SpMV
// launches (lss.hip) and the Krylov kernels that fuse a dot product into the product (krylov.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "lanes.hpp"

namespace cf3hip {
namespace spmv4 {

// Blocks a lane takes per trip of its row loop.  A block costs a chain of two loads (its column, then x), so the
// loads of a trip are issued together; positions past the row read its last block again and are not added.
// Where no row of the wave has more than kTail blocks left, they are taken one per lane and trip: loads that
// are not added would cost more than the latency.  Measured, one block per trip / always four / this, us:
// FP64 64^3 and 100^3 tetrahedra (15 blocks a row) 116, 418 / 104, 380 / 104, 380; 80^3 hexahedra (27) 375 / 354 / 341;
// 4 M blocks in rows of 1, 2, 4, 9: 280, 156, 125, 117 / 442, 246, 143, 126 / 277, 155, 124, 108.  FP32 54, 228 / 46, 200 / 45, 200;
// 203 / 182 / 181; rows of 1, 5, 9, 17: 251, 72, 63, 54 / 453, 103, 68, 56 / 248, 72, 64, 46.
constexpr int kTrip = 4;
constexpr uint32_t kTail64 = 4, kTail32 = 9;   // of 2 and 4 blocks side by side

// FP64 values: lanes 0-7 take block 2k, lanes 8-15 block 2k+1; lane l streams 2 consecutive doubles
// (16 B) of block row (l & 7) >> 1, columns 2 (l & 1) .. +1.  After the call, lanes with
// l < 8 and even l hold y[row * 4 + (l >> 1)]; `a` receives that component.
__device__ __forceinline__ double row_f64(const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ cols,
                                          const double* __restrict__ vals, const double* __restrict__ x, uint32_t row,
                                          int l, int& a, bool& out)
{
  const uint32_t q0 = row_ptr[row], q1 = row_ptr[row + 1];
  const int sub = l >> 3, li = l & 7;
  double acc = 0.;
  uint32_t q = q0 + sub;
  for(; q < q1 && __any(q1 - q > kTail64); q += 2 * kTrip) {
    double2 v[kTrip], xv[kTrip];
#pragma unroll
    for(int k = 0; k < kTrip; ++k) {
      const uint32_t qq = min(q + 2u * k, q1 - 1);
      v[k] = *reinterpret_cast<const double2*>(vals + (uint64_t)qq * 16 + 2 * li);
      xv[k] = *reinterpret_cast<const double2*>(x + (uint64_t)cols[qq] * 4 + 2 * (li & 1));
    }
#pragma unroll
    for(int k = 0; k < kTrip; ++k) {
      const double s = v[k].x * xv[k].x + v[k].y * xv[k].y;
      acc = q + 2u * k < q1 ? acc + s : acc;
    }
  }
  for(; q < q1; q += 2) {
    const double2 v = *reinterpret_cast<const double2*>(vals + (uint64_t)q * 16 + 2 * li);
    const double2 xv = *reinterpret_cast<const double2*>(x + (uint64_t)cols[q] * 4 + 2 * (li & 1));
    acc += v.x * xv.x + v.y * xv.y;
  }
  acc += lanes::move<lanes::kXor1>(acc);
  acc += lanes::move<lanes::kNext8>(acc);
  a = li >> 1;
  out = l < 8 && (l & 1) == 0;
  return acc;
}

// FP32 values, FP64 vectors and accumulation: lane l streams one block row (4 floats, 16 B) of
// blocks 4k + (l >> 2), component l & 3; lanes l < 4 hold y[row * 4 + l] after the call.
// One block per trip: with 12 doubles a block in flight, four cost more waves than they hide latency.  Per iteration of
// the precision form (two products and the vector kernels), four -> two -> one, us: 100^3 tetrahedra 746 -> 725 -> 694;
// hexahedra 100^3 1308 with two, 1220 with one; 37^3 and 60^3 tetrahedra equal within 1 %.
__device__ __forceinline__ double row_mixed(const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ cols,
                                            const float* __restrict__ vals, const double* __restrict__ x,
                                            uint32_t row, int l, int& a, bool& out)
{
  const uint32_t q0 = row_ptr[row], q1 = row_ptr[row + 1];
  const int sub = l >> 2;
  a = l & 3;
  double acc = 0.;
  for(uint32_t q = q0 + sub; q < q1; q += 4) {
    const double2* xb = reinterpret_cast<const double2*>(x + (uint64_t)cols[q] * 4);
    const float4 v = *reinterpret_cast<const float4*>(vals + (uint64_t)q * 16 + 4 * a);
    const double2 x01 = xb[0], x23 = xb[1];
    acc += (double)v.x * x01.x + (double)v.y * x01.y + (double)v.z * x23.x + (double)v.w * x23.y;
  }
  acc += lanes::move<lanes::kNext4>(acc);
  acc += lanes::move<lanes::kNext8>(acc);
  out = l < 4;
  return acc;
}

// FP32 values and vectors, FP32 accumulation (lane layout of row_mixed): the inner product of the
// precision form with FP32 vectors
__device__ __forceinline__ float row_f32(const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ cols,
                                         const float* __restrict__ vals, const float* __restrict__ x, uint32_t row,
                                         int l, int& a, bool& out)
{
  const uint32_t q0 = row_ptr[row], q1 = row_ptr[row + 1];
  const int sub = l >> 2;
  a = l & 3;
  float acc = 0.f;
  uint32_t q = q0 + sub;
  for(; q < q1 && __any(q1 - q > kTail32); q += 4 * kTrip) {
    float4 v[kTrip], xv[kTrip];
#pragma unroll
    for(int k = 0; k < kTrip; ++k) {
      const uint32_t qq = min(q + 4u * k, q1 - 1);
      v[k] = *reinterpret_cast<const float4*>(vals + (uint64_t)qq * 16 + 4 * a);
      xv[k] = *reinterpret_cast<const float4*>(x + (uint64_t)cols[qq] * 4);
    }
#pragma unroll
    for(int k = 0; k < kTrip; ++k) {
      const float s = v[k].x * xv[k].x + v[k].y * xv[k].y + v[k].z * xv[k].z + v[k].w * xv[k].w;
      acc = q + 4u * k < q1 ? acc + s : acc;
    }
  }
  for(; q < q1; q += 4) {
    const float4 v = *reinterpret_cast<const float4*>(vals + (uint64_t)q * 16 + 4 * a);
    const float4 xv = *reinterpret_cast<const float4*>(x + (uint64_t)cols[q] * 4);
    acc += v.x * xv.x + v.y * xv.y + v.z * xv.z + v.w * xv.w;
  }
  acc += lanes::move<lanes::kNext4>(acc);
  acc += lanes::move<lanes::kNext8>(acc);
  out = l < 4;
  return acc;
}

template<typename VR>
__device__ __forceinline__ double row(const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ cols,
                                      const VR* __restrict__ vals, const double* __restrict__ x, uint32_t r, int l,
                                      int& a, bool& out)
{
  if constexpr(sizeof(VR) == sizeof(double)) return row_f64(row_ptr, cols, vals, x, r, l, a, out);
  else return row_mixed(row_ptr, cols, vals, x, r, l, a, out);
}

}  // namespace spmv4
}  // namespace cf3hip
