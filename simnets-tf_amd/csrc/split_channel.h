// Which channel a staging lane of the input gradient's split kernel reads (similarity_split.hip): plain C++, also compiled by the
// host-side tests.  A chunk holds one or two groups of eight channels; a lane's address starts at its group's first channel in
// chunk 0 and a uniform offset, unsigned, leads from there.  Channels behind the last are read as the last.
#pragma once

#include "fast_div.h"

namespace simnets {

// The channel at which the addresses of group g start: the first one's where eight channels or fewer have no second group, in
// chunks of sixteen (its values are not used: an offset back from it to the last channel would be negative).
SIMNETS_HOST_DEVICE int split_group_start(int C, int g) { return C > 8 ? 8 * g : 0; }

// From there, value j's channel in the chunk that starts at channel `first`: at least 0, and C - 1 - start at most.
SIMNETS_HOST_DEVICE int split_channel_offset(int C, int start, int first, int j)
{
    const int there = C - 1 - (first + start);
    return first + (there < j ? (there < -start ? -start : there) : j);
}

}  // namespace simnets
