// Device descriptor arrays handed over by the caller: who reads them.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace v3dm {

// Whether the row kernel reads the caller's `bytes` at src itself.  It has none of the copy
// engine's checks, so the array must be memory of the handle's own device (ownDevice), lie whole
// inside its allocation [base, base + size), apart from the set's buffer dst, and be aligned for
// the kernel's 8-byte loads.  Any other pointer goes through a copy, which takes it or refuses it.
inline bool rows_readable(uintptr_t src, size_t bytes, bool ownDevice, uintptr_t base, size_t size, uintptr_t dst)
{
    bool const inside = src >= base && src - base <= size && bytes <= size - (src - base);
    bool const apart = src + bytes <= dst || dst + bytes <= src;
    return ownDevice && inside && apart && (src & 7) == 0;
}

}  // namespace v3dm
