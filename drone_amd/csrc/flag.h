// Waiting for a stream by way of a word of pinned memory that its last kernel writes.
//
// hipStreamSynchronize takes 4 us longer than the host needs to see such a word, the launch of a kernel that does nothing else
// included (a kernel and a wait 15.7 / 11.7 us on one stream, 10.9 where the kernel writes the word itself), and a superstep, a traversal or an
// epoch waits once or more.  The kernels of a stream start one after the other, each behind the release of all that the one before
// wrote, so when a kernel writes the word everything that was enqueued before that kernel is done and visible, to other streams and copies
// too.  What the writing kernel itself stores to device memory is not: such a kernel is followed by raise_flag_kernel.
#pragma once
#include "common.h"

namespace drone {

__device__ __forceinline__ void raise_flag(unsigned *word, unsigned value)
{
    __hip_atomic_store(word, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);  // behind this thread's other stores
}

// Returns when the kernel that writes f->raised has done so, or an error of the stream.
hipError_t flag_seen(drone_flag *f, hipStream_t s);
// The same for everything that has been enqueued.
hipError_t flag_wait(drone_flag *f, hipStream_t s);

}  // namespace drone
