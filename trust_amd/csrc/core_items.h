// Sizes of the dense core's work items (core.hip).
#pragma once

namespace trust {

constexpr int kCorePart = 2048;  // dense targets per work item (longer lists are cut)

// Slots of the item list for `rows` candidate rows out of E entries.  Every
// candidate row takes one from the back; one with nd > kCorePart targets also
// takes ceil(nd / kCorePart) < 2 nd / kCorePart from the front, and the rows'
// targets are at most E together.
inline long long core_item_slots(long long rows, long long E)
{
    return rows + 2 * E / kCorePart;
}

}  // namespace trust
