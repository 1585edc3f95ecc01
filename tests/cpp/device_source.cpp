// rows_readable (csrc/v3dm_source.h) at the edges of an allocation and of the set's buffer.
#include <cstdio>

#include "../../eth-v3d-lgpl_amd/csrc/v3dm_source.h"

static int bad = 0;

static void expect(char const* what, bool got, bool want)
{
    if (got != want) {
        std::printf("%s: %d, expected %d\n", what, got, want);
        bad = 1;
    }
}

int main()
{
    using v3dm::rows_readable;
    uintptr_t const base = 0x10000, dst = 0x900000;
    size_t const size = 4096;
    expect("whole", rows_readable(base, size, true, base, size, dst), true);
    expect("tail", rows_readable(base + 1024, size - 1024, true, base, size, dst), true);
    expect("one row too many", rows_readable(base, size + 512, true, base, size, dst), false);
    expect("from the middle past the end", rows_readable(base + 1024, size, true, base, size, dst), false);
    expect("before the allocation", rows_readable(base - 512, 512, true, base, size, dst), false);
    expect("past the allocation", rows_readable(base + size + 512, 512, true, base, size, dst), false);
    expect("empty at the end", rows_readable(base + size, 0, true, base, size, dst), true);
    expect("other memory", rows_readable(base, size, false, base, size, dst), false);
    expect("odd address", rows_readable(base + 4, 512, true, base, size, dst), false);
    expect("the set's own buffer", rows_readable(dst, 512, true, dst, size, dst), false);
    expect("overlapping it", rows_readable(dst - 256, 512, true, dst - 1024, size, dst), false);
    expect("just below it", rows_readable(dst - 512, 512, true, dst - 1024, size, dst), true);
    expect("just above it", rows_readable(dst + 512, 512, true, dst, size, dst), true);
    return bad;
}
