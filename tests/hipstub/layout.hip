// Where the host code's tests find what they read and write.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <cstring>

#include "rast_launch.h"

extern "C" size_t layout_counters_size() { return sizeof(rast::FrameCounters); }

// The byte offset of a frame counter (SIZE_MAX: there is none of that name).
extern "C" size_t layout_counter(const char *name)
{
    using F = rast::FrameCounters;
#define FIELD(f) \
    if (!strcmp(name, #f)) return offsetof(F, f);
    FIELD(num_big) FIELD(total_pairs) FIELD(overflow_tiles) FIELD(ovf_entries) FIELD(pool_used) FIELD(storage_overflow)
    FIELD(capacity_wanted) FIELD(spilled) FIELD(past_fixed) FIELD(past_spill)
#undef FIELD
    return SIZE_MAX;
}
