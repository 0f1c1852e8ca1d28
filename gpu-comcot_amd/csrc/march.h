// What the marching kernels (march.hip, march_nl.hip) share: a wavefront
// holds a strip of 64 columns, one per lane, and marches along J with its
// rows in registers.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "comcot_consts.h"
#include "kernels.h"

namespace gc {

constexpr int kWave = 64;
constexpr int kMarchBlock = 256;

// Value of the lane one column to the west (I - 1) / east (I + 1); the
// outermost lane of the wave gets 0 (its results are never stored).
__device__ __forceinline__ float west(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float east(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}

// Planes are read and written through one buffer descriptor over the
// layer's block (every plane of a layer lies in one allocation, behind its
// depth plane): a lane's column is the vector offset, plane and row the
// scalar one, so rows cost no per-lane address arithmetic.  A lane that has
// nothing to store gives offset kNoStore, which the descriptor's range check
// drops: the row loop has no branch around a store.  (With branches the
// compiler has to assume the shorter path when it counts outstanding memory
// operations, and a wait for the next row's loads then also waits for
// stores.)
typedef __amdgpu_buffer_rsrc_t Block;
constexpr int kNoStore = -1;
__device__ __forceinline__ Block block_of(const DevLayer &L) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(L.h), 0, (int)L.block_bytes, 0x00027000);
}
__device__ __forceinline__ unsigned plane_off(const DevLayer &L, const void *p) {
  return (unsigned)(reinterpret_cast<unsigned long long>(p) -
                    reinterpret_cast<unsigned long long>(L.h));
}
__device__ __forceinline__ float get(Block b, int voff, unsigned soff) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b, voff, (int)soff, 0));
}
template <bool ST>
__device__ __forceinline__ void put(Block b, int voff, unsigned soff, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), b, voff, (int)soff, ST ? 2 : 0);
}

// A lane mask held in scalar registers as this lane's condition.
__device__ __forceinline__ bool lanes(unsigned long long m) {
  return __builtin_amdgcn_inverse_ballot_w64(m);
}

// Work of one wave: the first column and the rows j0..j1 it writes.
struct Strip {
  int c0, j0, j1;
};

// Group g of the row coefficients of row j (kRowCoef), by one scalar load
// (constant address space: nothing writes the table while kernels run).
typedef float Row4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ Row4 row_coef(const DevLayer &L, int j, int g) {
  typedef const __attribute__((address_space(4))) Row4 *ConstPtr;
  const int q = (j < 1 ? 1 : (j > L.ny ? L.ny : j)) - 1;
  return ((ConstPtr)(unsigned long long)L.rowc)[(size_t)q * (kRowCoef / 4) + g];
}

// OPEN (boundaries.f90:22-202) at one ring cell: a, b are the two flux
// components it combines (an average along the edge or a corner's own
// flux, and the flux across), cc = sqrt(g H), neg says which way the wave
// leaves.
__device__ __forceinline__ float radiate(float h, float cc, float a, float b, bool neg) {
  float zz = sqrtf(a * a + b * b) / cc;
  if (neg) zz = -zz;
  if (fabsf(zz) > kUB) zz = 0.0f;
  return h > kGx ? zz : 0.0f;
}

// Gauge sample (GET_TS, output.f90:1085-1094): the 2x2 stencil of the
// elevation weighted in the Fortran's operation order.
__device__ __forceinline__ float gauge_sample(const GaugeDev &G, const float *z) {
  const size_t o = (size_t)(G.kj - 1) * G.nx + (G.ki - 1);
  const float l1 = z[o], l2 = z[o + 1], l3 = z[o + G.nx], l4 = z[o + G.nx + 1];
  const float z1 = l1 * (1.0f - G.cx) * (1.0f - G.cy);
  const float z2 = l2 * G.cx * (1.0f - G.cy);
  const float z3 = l3 * (1.0f - G.cx) * G.cy;
  const float z4 = l4 * G.cx * G.cy;
  float dat = z1 + z2 + z3 + z4;
  if (fabsf(G.tide) > kGx) dat = dat + G.tide;
  return dat;
}

// The gauges of the step before ride in a step's launch (DevLayer::gauges; a
// launch of their own takes 4.5 us a step): workgroup 0 samples them, first,
// so that its chain of loads ends with the tiles', and seven idle ones keep
// the others on their XCDs.  step_block: this workgroup's number among the
// step's own, -1 for those eight.
inline int gauge_blocks(const DevLayer &L) { return L.ngauge > 0 ? 8 : 0; }
__device__ __forceinline__ int step_block(const DevLayer &L) {
  const int b = blockIdx.x;
  if (L.ngauge == 0) return b;
  if (b == 0) {
    const int step = L.ctl[L.ctl_in];
    for (int k = threadIdx.x; k < L.ngauge; k += blockDim.x)
      L.gauge_ring[(size_t)k * L.gauge_cap + (step - 1) % L.gauge_cap] = gauge_sample(L.gauges[k], L.z1);
  }
  return b < 8 ? -1 : b - 8;
}

}  // namespace gc
