// Waiting for a stream by way of a word of pinned memory that a last kernel writes.
//
// hipStreamSynchronize takes 4 us longer than the host needs to see such a word, the launch of a kernel that does nothing else
// included (a kernel and a wait 15.7 / 11.7 us on one stream), and a superstep or an epoch waits once or more.  The kernels of a stream start one
// after the other, each behind the release of all that the one before wrote, so when a kernel writes the word everything that was
// enqueued before that kernel is done and visible, to other streams and copies too.
//
// The runtime does not learn of it, and its next copy or launch on another stream waits for the stream on its own account: a
// traversal's call alone is 4 us faster so, but a call and a copy of its labels to the host 25 us slower (500,009 vertices 95 -> 127 us,
// distances over 1 M 215 -> 247).  So only calls that usually follow each other wait this way (ten supersteps 680 -> 635 us, with a copy of the
// ranks behind them 751 / 751; an epoch and its evaluation 142 -> 135, with a copy of the weights 160 / 151).
#pragma once
#include "common.h"

namespace drone {

// Returns when everything that has been enqueued is done, or an error of the stream.
hipError_t flag_wait(drone_flag *f, hipStream_t s);

}  // namespace drone
