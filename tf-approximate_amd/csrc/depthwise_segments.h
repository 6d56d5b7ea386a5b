// How a depthwise window kernel cuts output rows into column segments (host code without any of HIP's).
#pragma once
#include <cstdint>

namespace axc {

struct Segments {
    int count, length;   // the last one may be shorter
};

// The segments of ow columns for which cost(count, length) is least (negative: not possible), the fewest of equals; one segment
// if none is possible.  Counts with the same length are one choice, so only the first count of every length is looked at: some
// 2 sqrt(ow) of them (every count, of a row of 32 767 columns, took 125 us of a call).
template <typename Cost>
Segments best_segments(const int ow, Cost &&cost)
{
    Segments best = {1, ow};
    int64_t least = -1;
    for (int count = 1; count <= ow;) {
        const int length = (ow + count - 1) / count;
        const int64_t c = cost((ow + length - 1) / length, length);
        if (c >= 0 && (least < 0 || c < least)) {
            least = c;
            best = {(ow + length - 1) / length, length};
        }
        if (length == 1)
            break;
        count = (ow + length - 2) / (length - 1);   // the first whose length is smaller
    }
    return best;
}

} // namespace axc
