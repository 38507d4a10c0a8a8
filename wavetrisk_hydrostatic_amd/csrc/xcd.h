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

// Rows of a compute list's blocks per XCD for list_block, or 0 for the blocks as
// they come; planes: fields that the launch takes over the list (layers or
// members).  Measured, us a launch, as they come -> in rows: BiCGSTAB's applies
// at J8 32 -> 30 and 30 -> 26, Jacobi sweep at J8 27.7 -> 26.3, edge fluxes of
// J8 L30 209 -> 191 and of J7 L20 26 -> 22, odd prolongation at J7 L20 33 -> 27.
// Shorter launches lose by it, since the halo copies at the list's end fall to
// one XCD: at J7 (660 blocks) a sweep of one field 9.3 -> 11.5 and an apply 18.6
// -> 20.4 (an apply of three members 15.8 -> 15.5), at J6 (165) the applies of
// four members 8.3 -> 9.2 and 9.0 -> 10.3.  The host decides: the launch's size
// read in the kernel instead costs a sweep at J4 to J7 3 to 5 %.
// Not for the multi-level even prolongation, which reads several planes of two
// levels and loses at J8 (153 -> 206 us on the levels of J5 to J8 with L30).
inline int xcd_rows(unsigned blocks, int planes) {
  return blocks >= 512 && (unsigned long long)blocks * planes >= 1024 ? (int)(blocks / 8) : 0;
}
__device__ __forceinline__ unsigned list_block(unsigned per) {
  const unsigned b = blockIdx.x;
  return b < 8 * per ? b % 8 * per + b / 8 : b;
}
