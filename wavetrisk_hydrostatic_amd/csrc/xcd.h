// Blocks of a stencil in rows per XCD.
#pragma once
#include <hip/hip_runtime.h>

// The blocks of a launch are dealt to the eight XCDs in turn, and each XCD has
// an L2 of its own: neighbouring rows of a grid, some blocks apart, are then
// read from memory by several of them.  This order of the blocks gives every
// XCD an unbroken eighth of them (the rest of less than eight blocks stays
// where it is).
__device__ __forceinline__ unsigned xcd_block() {
  const unsigned per = gridDim.x / 8, b = blockIdx.x;
  return b < 8 * per ? b % 8 * per + b / 8 : b;
}

// the block of a compute list: in that order from 512 blocks (J7) on.  BiCGSTAB's
// applies at J8 32 -> 30 and 30 -> 26 us, edge fluxes of J8 L30 209 -> 191, odd
// prolongation at J7 L20 33 -> 27, an apply at J7 for three members 15.8 ->
// 15.5; below, an eighth is a few blocks and the halo copies at the list's end
// fall to one XCD: the applies at J6 for four members 8.3 -> 9.2 and 9.0 -> 10.3.
// Not for the multi-level even prolongation, which reads several planes of two
// levels and loses at J8 (153 -> 206 us on the levels of J5 to J8 with L30).
__device__ __forceinline__ unsigned list_block() { return gridDim.x < 512 ? blockIdx.x : xcd_block(); }
