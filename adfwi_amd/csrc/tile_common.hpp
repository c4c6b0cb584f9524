// What the register-tile kernels share (included by acoustic_tile.hpp and elastic_tile.hpp, inside their
// files' namespace).
#pragma once

namespace tile {

// value of the lane one to the left / right (0 past the wavefront's ends, which only halo
// columns see)
__device__ __forceinline__ float from_left(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float from_right(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
}

// the exchange between wavefronts goes through LDS only: loads and stores of global memory may
// stay in flight across it
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// a value no kernel writes, at a wave-uniform address: a scalar load, outside the vector
// memory queue (a vector load here would make the wave wait for every prefetch issued before it)
template <class T>
__device__ __forceinline__ T scalar_ld(const T *p) {
  return *(const __attribute__((address_space(4))) T *)(unsigned long long)p;
}

// forms the values where this stands: left to itself the compiler moves a sum whose only use lies past
// a later branch there, and holds its terms till then
__device__ __forceinline__ void pin(float &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin(float &a, float &b) { asm volatile("" : "+v"(a), "+v"(b)); }

// workgroup -> (tile, group of shots): blocks go round-robin to the 8 XCDs, and every XCD takes a
// contiguous run of a group's tiles, row by row, so that its L2 serves the halos neighbouring tiles
// share and joins the ends of their rows, which share cache lines, before they are written back.
// (With the groups of one tile next to each other instead, for the sake of its coefficients, us per step:
// acoustic forward 136 against 128 and adjoint 190 against 168 on 464 x 1232 with 64 shots; elastic forward
// with a trace 135 against 108 on 242 x 680 / 32 shots, 464 against 362 on 362 x 1040 / 48.)
template <class G>
__device__ __forceinline__ void place(const G &g, int &tx, int &tz, int &grp) {
  const int n = (int)gridDim.x, b = (int)blockIdx.x;
  const int xcd = b & 7, per = n >> 3, rem = n & 7;
  const int logical = xcd * per + min(xcd, rem) + (b >> 3);
  const int nt = g.ntx * g.ntz;
  grp = logical / nt;
  const int tl = logical - grp * nt;
  tz = tl / g.ntx;
  tx = tl - tz * g.ntx;
}

}  // namespace tile
