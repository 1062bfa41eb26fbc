// The elements of a plane that one of the LANES lanes sharing it adds, in order: lane, lane + LANES, ...
// below `count`, AHEAD at a time (batch(i): i, i + LANES, ..., all within the plane), then singly
// (one(i)). The index is unsigned: count may be 2^31 - 1, and the step past it does not fit an int.
#pragma once

namespace mfh {

template <unsigned LANES, unsigned AHEAD, class Batch, class One>
__host__ __device__ inline void walk_plane(unsigned lane, unsigned count, Batch batch, One one) {
    unsigned i = lane;
    for (; i + (AHEAD - 1) * LANES < count; i += AHEAD * LANES) batch(i);
    for (; i < count; i += LANES) one(i);
}

}  // namespace mfh
