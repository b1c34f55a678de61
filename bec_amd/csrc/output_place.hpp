// Where a kernel may write a caller's output itself instead of copying it there.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace bec {

// What the runtime says of an output pointer: whether it is device memory, of which
// device, and the allocation it lies in.
struct OutputPlace {
    bool device_memory = false;
    int device = -1;
    uintptr_t base = 0;
    size_t size = 0;
};

// Device memory of the writer's own device that holds all of the output, apart from
// the input.  Everything else takes the copy: a kernel may not reach another device's
// memory (a fault without peer access), writes host memory one store at a time, and
// an output that overlaps the input partly would be checked against the input's size.
inline bool writes_direct(const OutputPlace &p, int own_device, uintptr_t y, size_t bytes, uintptr_t x, size_t x_bytes)
{
    if (!p.device_memory || p.device != own_device || y % sizeof(float) != 0) return false;
    if (y < p.base || y - p.base > p.size || bytes > p.size - (y - p.base)) return false;
    return y >= x ? y - x >= x_bytes : x - y >= bytes;
}

} // namespace bec
