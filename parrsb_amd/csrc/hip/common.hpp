// Shared device helpers for the gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define RSB_WAVE 64

// Order-preserving map of an IEEE double to uint64 (total order equal to `<`
// on non-NaN values, with -0.0 mapped onto +0.0 so they compare equal, as
// C's `<` has them).
__host__ __device__ inline uint64_t dkey(double x) {
  if (x == 0.0) x = 0.0;
  uint64_t u;
  __builtin_memcpy(&u, &x, 8);
  return (u & 0x8000000000000000ull) ? ~u : (u | 0x8000000000000000ull);
}
__host__ __device__ inline double dkey_inv(uint64_t k) {
  uint64_t u = (k & 0x8000000000000000ull) ? (k & 0x7fffffffffffffffull) : ~k;
  double x;
  __builtin_memcpy(&x, &u, 8);
  return x;
}
__host__ __device__ inline uint32_t fkey(float x) {
  if (x == 0.0f) x = 0.0f;
  uint32_t u;
  __builtin_memcpy(&u, &x, 4);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Sum over the wave by butterflies of distance 32, 16, 8, 4, 2, 1, every
// step on the VALU: half- and row-swaps for 32 and 16, then (the values
// being periodic with the last distance) row rotations by 8 and 4 and quad
// permutations reach the same partner as an exclusive-or of the lane number,
// so the result has the bits of the same butterflies through LDS permutes,
// which took a round trip a step.
__device__ inline unsigned wave_swap32(unsigned v, unsigned &other) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  other = r[1];
  return r[0];
}
__device__ inline unsigned wave_swap16(unsigned v, unsigned &other) {
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  other = r[1];
  return r[0];
}
template <int CTRL>
__device__ inline unsigned wave_dpp(unsigned v) {
  return (unsigned)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}
template <int STEP, typename T>
__device__ inline T wave_step(T v) {
  constexpr int NW = sizeof(T) / 4;
  unsigned w[NW], x[NW], y[NW];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (int i = 0; i < NW; i++) {
    if (STEP == 32) x[i] = wave_swap32(w[i], y[i]);
    else if (STEP == 16) x[i] = wave_swap16(w[i], y[i]);
    else x[i] = w[i];
    if (STEP == 8) y[i] = wave_dpp<0x128>(w[i]);  // row_ror:8
    if (STEP == 4) y[i] = wave_dpp<0x124>(w[i]);  // row_ror:4
    if (STEP == 2) y[i] = wave_dpp<0x4e>(w[i]);   // quad_perm [2,3,0,1]
    if (STEP == 1) y[i] = wave_dpp<0xb1>(w[i]);   // quad_perm [1,0,3,2]
  }
  T a, b;
  __builtin_memcpy(&a, x, sizeof(T));
  __builtin_memcpy(&b, y, sizeof(T));
  return a + b;
}
template <typename T>
__device__ inline T wave_sum(T v) {
  static_assert(sizeof(T) == 4 || sizeof(T) == 8, "whole words");
  v = wave_step<32>(v);
  v = wave_step<16>(v);
  v = wave_step<8>(v);
  v = wave_step<4>(v);
  v = wave_step<2>(v);
  return wave_step<1>(v);
}

// Block-wide sum of NV doubles with a fixed reduction tree (deterministic).
// `red` must hold (blockDim.x / 64) * NV doubles.  Result valid in thread 0.
// NW: waves per workgroup where the kernel knows it (0: from blockDim).
template <int NV, int NW = 0>
__device__ inline void block_sum(double (&v)[NV], double *red) {
  const int lane = threadIdx.x & (RSB_WAVE - 1), wid = threadIdx.x / RSB_WAVE;
  const int nw = NW ? NW : blockDim.x / RSB_WAVE;
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = wave_sum(v[k]);
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < NV; k++) red[wid * NV + k] = v[k];
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      double s = red[k];
#pragma unroll(NW ? NW : 1)
      for (int w = 1; w < nw; w++) s += red[w * NV + k];
      v[k] = s;
    }
  }
  __syncthreads();
}

