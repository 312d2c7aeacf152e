// cv_reads.h -- which bytes a kernel reads of a batch of vectors of any length.  A lane reads its k-slots 16, 8 or 4 bytes at a time at
// whatever element they begin; what it gets of the elements behind its slice is cleared in registers, but no read may touch a byte behind the
// last vector.  Without HIP, so that every read can be checked against its buffer on the host.  Offsets and ends are bytes from the first vector.
#pragma once
#include "cv_layout.h"

namespace cv {

// bytes from the first vector's first to the last one's last
CV_HD uint64_t vectorsEnd(uint32_t batch, uint64_t stride, uint32_t in, uint32_t esz) { return (uint64_t)(batch - 1u) * stride + (uint64_t)in * esz; }

// bytes of lane group g's slice (gs k-slots to a group) that exist
CV_HD int32_t sliceBytes(uint32_t in, uint32_t gs, uint32_t g, uint32_t esz)
{
    const int32_t left = (int32_t)in - (int32_t)(g * gs), some = left > 0 ? left : 0;
    return (some < (int32_t)gs ? some : (int32_t)gs) * (int32_t)esz;
}

// Where the reads of `samples` vectors from vector `first` on end at most: those of the last lane group, whose fragments hold `slots` k-slots.
CV_HD uint64_t tileReadsEnd(uint64_t first, uint32_t samples, uint64_t stride, uint32_t gs, uint32_t slots, uint32_t esz)
{
    return (first + samples - 1u) * stride + (uint64_t)(3u * gs + slots) * esz;
}

// A read of `bytes` bytes that is wanted at `want`, of vectors that end at `end` (at least `bytes` behind the first; addresses or offsets): where it is
// made, and by how many bytes what it brings is moved down then (all of it, where nothing that is wanted exists).
template <typename At>
CV_HD At readAt(At want, uint32_t bytes, At end)
{
    static_assert(sizeof(At) == 8, "differences are taken as signed 64-bit numbers");
    return (int64_t)(want + bytes - end) > 0 ? end - bytes : want;
}
template <typename At>
CV_HD uint32_t readDown(At want, uint32_t bytes, At end)
{
    static_assert(sizeof(At) == 8, "differences are taken as signed 64-bit numbers");
    const int64_t over = (int64_t)(want + bytes - end);
    return over < 0 ? 0u : over > (int64_t)bytes ? bytes : (uint32_t)over;
}

} // namespace cv
