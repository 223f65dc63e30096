// host_rules.h -- host-side rules that need neither HIP nor a device.
#pragma once

#include <stddef.h>

#include <initializer_list>

namespace skm {

// A workspace of several buffers: grab(&p, bytes) each (0 or an error code),
// or none of them -- after a failure the ones already there are dropped and
// null, so that a later call sees no half of a workspace.
struct Buffer {
    void** p;
    size_t bytes;
};
template <typename Grab, typename Drop>
int grab_all(std::initializer_list<Buffer> list, Grab grab, Drop drop)
{
    for (const Buffer* b = list.begin(); b != list.end(); ++b) {
        const int rc = grab(b->p, b->bytes);
        if (rc == 0) continue;
        *b->p = nullptr;
        while (b != list.begin()) {
            --b;
            drop(*b->p);
            *b->p = nullptr;
        }
        return rc;
    }
    return 0;
}

// Rows that one launch of k_screen_wide takes: their two largest values of
// every 128 centres, 16 bytes a row and 256 centres, stay under kWidePartBytes
// (a launch then has at most 65,536 blocks, 256 rounds of the CUs: what a
// launch costs and the round that it leaves partly idle are lost in them).
// All rows at once would take 8 times X for 65,536 centres of 132 floats, and
// from 8.4M blocks of 512 threads a launch is refused.
constexpr size_t kWidePartBytes = size_t(256) << 20;
inline long wide_rows(long n, int k)
{
    const long ncg = (k + 255) / 256;
    const long rows = (long)(kWidePartBytes / size_t(16 * ncg)) / 2048 * 2048;  // 256 for each of 8 XCDs
    return n < rows ? n : rows < 2048 ? 2048 : rows;
}
inline size_t wide_part_floats(long rows, int k) { return size_t(rows) * ((size_t(k) + 255) / 256) * 4; }
// k_screen_wide's blocks for `rows` rows: whole turns of the XCDs.
inline long wide_blocks(long rows, int k) { return ((rows + 255) / 256 + 7) / 8 * 8 * ((k + 255) / 256); }

}  // namespace skm
