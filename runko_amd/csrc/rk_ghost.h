// Ghost images of an interior node of a periodic lattice.
//
// On a world with at least 2 * HALO cells along every axis a node has at most
// one image in the ghost shell along an axis.  Offsets are unsigned, modulo
// 2^32 as the lattice's indices: on a lattice of 2^31 nodes and more a single
// step along x is past what an int holds.  Plain functions, so that the host can
// check them.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#define RK_GHOST_FN __host__ __device__ inline
#else
#define RK_GHOST_FN inline
#endif

namespace rk {

constexpr int GHOST_LAYERS = 3;

// cells from interior coordinate c (from GHOST_LAYERS on, of N) to its image; 0: it has none
RK_GHOST_FN uint32_t ghost_step(int c, int N)
{
  return c < 2 * GHOST_LAYERS ? uint32_t(N) : (c >= N ? uint32_t(-N) : 0u);
}

// the same along axis 0 or 1 as an offset in a lattice of L nodes per axis
RK_GHOST_FN uint32_t ghost_row(const int N[3], const int L[3], int c, int axis)
{
  const uint32_t row = axis == 0 ? uint32_t(L[1]) * uint32_t(L[2]) : uint32_t(L[2]);
  return ghost_step(c, N[axis]) * row;
}

// image n (bits 4, 2, 1: displaced along axis 0, 1, 2) from its node, and
// whether a node with these displacements has it
RK_GHOST_FN uint32_t ghost_image(int n, uint32_t d0, uint32_t d1, uint32_t d2)
{
  return (n & 4 ? d0 : 0u) + (n & 2 ? d1 : 0u) + (n & 1 ? d2 : 0u);
}
RK_GHOST_FN bool ghost_there(int n, uint32_t d0, uint32_t d1, uint32_t d2)
{
  return (!(n & 4) || d0 != 0) && (!(n & 2) || d1 != 0) && (!(n & 1) || d2 != 0);
}

}  // namespace rk
