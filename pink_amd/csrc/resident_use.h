// Which resident launches of a device may run at once (see launch_resident).
#pragma once
#include <cstddef>
#include <cstdint>

// A launch's blocks, and how many of them a compute unit holds.
struct ResidentShape {
    uint32_t blocks, per_unit;
};

// How many of the `count` launches in flight, oldest first, a new one has to wait for: so many that every block of what is left
// and of its own has a place on the device at once.  What counts is the number of blocks that a unit holds of any of the kernels,
// the smallest of them: a unit has room for so many whichever they are.
template <typename Shapes>
size_t resident_waits(const Shapes &in_flight, size_t count, ResidentShape mine, uint32_t units)
{
    for (size_t first = 0;; ++first) {
        uint64_t blocks = mine.blocks;
        uint32_t per_unit = mine.per_unit;
        for (size_t i = first; i < count; ++i) {
            blocks += in_flight[i].blocks;
            per_unit = per_unit < in_flight[i].per_unit ? per_unit : in_flight[i].per_unit;
        }
        if (first == count || blocks <= (uint64_t)units * per_unit) return first;
    }
}
