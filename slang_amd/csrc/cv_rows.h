// cv_rows.h -- whether two regions of rows in memory meet.  Without HIP.
#pragma once
#include <stdint.h>

namespace cv {

// Whether two regions of `rows` rows each, `stride` bytes apart and `width` bytes wide, may have a byte in common (between their first
// and their last byte: rows of one in the gaps of the other count as well).
struct Rows { uint64_t at, stride, width; };
inline bool rowsMeet(const Rows& a, const Rows& b, uint32_t rows)
{
    const uint64_t aEnd = a.at + (rows - 1ull) * a.stride + a.width, bEnd = b.at + (rows - 1ull) * b.stride + b.width;
    return a.at < bEnd && b.at < aEnd;
}

// The same, but rows at one distance of which each lies in a gap of the other region's do not meet.
inline bool rowsOverlap(const Rows& a, const Rows& b, uint32_t rows)
{
    if (!rowsMeet(a, b, rows)) return false;
    if (a.stride != b.stride || a.stride == 0) return true;
    const uint64_t s = a.stride, d = b.at >= a.at ? (b.at - a.at) % s : (s - (a.at - b.at) % s) % s;
    return d < a.width || d + b.width > s;
}

} // namespace cv
