// Limits of one kernel launch.  Host code only.
#pragma once

namespace sw {

// A launch takes fewer than 2^32 threads along an axis.
constexpr long long kMaxLaunchThreads = (1ll << 32) - 1;

inline bool launch_fits(long long blocks, int threads)
{
    return blocks <= kMaxLaunchThreads / threads;
}

// Planes per z chunk of a z-marching launch that lays all its blocks (threads
// each) along one axis: `planes` as long as the chunks of `columns` columns of
// iz planes fit beside `more` other blocks, otherwise the next multiple of it
// by a power of two that does.
inline int z_chunk_planes(int planes, long long columns, int iz, int threads, long long more)
{
    while (planes < iz && !launch_fits(columns * ((iz + planes - 1) / planes) + more, threads))
        planes = planes > iz / 2 ? iz : 2 * planes;
    return planes;
}

}  // namespace sw
