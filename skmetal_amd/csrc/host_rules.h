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

}  // namespace skm
