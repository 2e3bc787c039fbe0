// Which of several workgroups is the last to arrive at a counter.
//
// The arrival number reaches the other waves through one word of LDS that the caller uses again right
// after.  So there are two barriers after it is written: the first makes it visible, the second ends only
// when every wave has read it (without that one a wave that is late to read finds what another has put
// there since, takes itself for one of an earlier workgroup and leaves).
//
// Written against an executor, so that the order of the waves can be forced on the CPU:
//   arrive()   this thread's earlier global atomics are performed; one thread then counts (leader)
//   barrier()  workgroup barrier
//   count()    the counter's value before this workgroup added one
//   put/get    the LDS word
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define CCA_ARRIVAL_HD __device__ __forceinline__
#else
#define CCA_ARRIVAL_HD inline
#endif

namespace cca {

template <class Ex>
CCA_ARRIVAL_HD bool last_of(const Ex& ex, uint32_t n) {
    ex.arrive();
    ex.barrier();
    if (ex.leader()) ex.put(ex.count());
    ex.barrier();
    const bool last = ex.get() == n - 1;
    ex.barrier();
    return last;
}

}  // namespace cca
