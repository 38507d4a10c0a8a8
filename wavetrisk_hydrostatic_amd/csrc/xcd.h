// Blocks of a stencil over a long list, in rows per XCD.
#pragma once
#include <hip/hip_runtime.h>

// The blocks of a launch are dealt to the eight XCDs in turn, and each XCD has
// an L2 of its own: neighbouring rows of a grid, some blocks apart in its list,
// are then read from memory by several of them.  This order of the blocks
// gives every XCD an unbroken eighth of the list (the rest of less than eight
// blocks stays where it is).  Measured with it: BiCGSTAB's applies at J8 32 -> 30
// and 30 -> 26 us, edge fluxes of J8 L30 209 -> 191 us, odd prolongation at J7
// L20 33 -> 27 us; the others' stencils 0 to 10 %.
__device__ __forceinline__ unsigned xcd_block() {
  const unsigned per = gridDim.x / 8, b = blockIdx.x;
  return b < 8 * per ? b % 8 * per + b / 8 : b;
}
