// How the lanes of a wave hand each other values through the wave's part of
// LDS (the emit's staging, the classify's list of active cells).
//
// The lanes run the same instruction together, but nothing in the language
// says that they do: a compiler may give lanes on two sides of a branch their
// own copies of what follows it and run the one to its end before the other.
// So every step that reads what other lanes wrote, or writes where other lanes
// may still read, stands behind `order`, which the kernels make a point that
// the wave passes together (no instruction: LDS serves a wave in order).
//
// Plain C++ (no HIP types) so that a host test can run the lanes one after the
// other between these points.
#ifndef MDMC_WAVE_H
#define MDMC_WAVE_H

#include <cstdint>

#if defined(__HIPCC__)
#define MDMC_LANE __host__ __device__ __attribute__((always_inline))
#else
#define MDMC_LANE
#endif

namespace mdmc {

// Every lane puts its words in the shared part, then copies out words that any
// lane may have put there.  What the part held before has been read when the
// first lane puts, and the copies are made when the part is used again.
template <class Put, class Copy, class Order>
MDMC_LANE inline void wave_exchange(Put put, Copy copy, Order order) {
  order();
  put();
  order();
  copy();
  order();
}

// Entry `first` + lane of a ring of N entries that any lanes filled, for the
// first n lanes (0 for the others).
template <uint32_t N, class Order>
MDMC_LANE inline uint32_t ring_take(const uint16_t *ring, uint32_t first, uint32_t lane, uint32_t n, Order order) {
  static_assert((N & (N - 1u)) == 0u, "a power of two");
  order();
  return lane < n ? ring[(first + lane) & (N - 1u)] : 0u;
}

}  // namespace mdmc

#endif
