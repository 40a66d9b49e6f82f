// Rules of the split order-1 tANS decoder that hold without a kernel (fz_entropy.hip has the kernels).
#pragma once
#include <stdint.h>

#ifndef FZ_HD
#ifdef __HIPCC__
#define FZ_HD __host__ __device__ inline
#else
#define FZ_HD inline
#endif
#endif

namespace fz {

// The nodes of all graph waves of a call go to one pool. Every wave of every round adds its number of
// nodes to one count, also when the pool is full, and 1,500 million codes with an escape in 20 make more
// than 2^32 of them (3 nodes a code): the count has 64 bits, so that a wave that finds the pool
// full keeps finding it full. First nodes are kept in 32 bits (all ones: no room).
typedef unsigned long long NodeCount;
constexpr uint32_t kPoolNone = ~0u;
constexpr uint64_t kPoolMax = 0xF0000000ull;
static_assert(kPoolMax < kPoolNone, "a first node is never taken for no room");

// Where a wave's nn nodes go when the count was `before`; kPoolNone: they do not fit.
FZ_HD uint32_t pool_first(NodeCount before, uint32_t nn, uint64_t cap) {
    return before + nn <= cap ? (uint32_t)before : kPoolNone;
}

}  // namespace fz
