// Where the host code's tests find what they read and write.
#include <hip/hip_runtime.h>

#include <cstddef>

#include "rast_launch.h"

extern "C" size_t layout_counters_size() { return sizeof(rast::FrameCounters); }

extern "C" size_t layout_counter(int k)
{
    using F = rast::FrameCounters;
    switch (k) {
    case 0: return offsetof(F, total_pairs);
    case 1: return offsetof(F, ovf_entries);
    case 2: return offsetof(F, pool_used);
    case 3: return offsetof(F, storage_overflow);
    case 4: return offsetof(F, spilled);
    default: return sizeof(F);
    }
}
