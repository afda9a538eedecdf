// Equal device buffers that a context keeps between calls, where some forms of a computation want more of
// them than others need.
#pragma once
#include <stddef.h>

namespace pa {

struct BufferSet {
    static constexpr int kMax = 5;
    void* p[kMax] = {};
    size_t cap = 0;    // bytes of each
    int n = 0;         // held
    int room = kMax;   // as many of cap bytes as fitted when more were asked for

    template <class Free> void clear(Free release) {
        for (int i = 0; i < n; ++i) release(p[i]);
        for (auto& q : p) q = nullptr;
        cap = 0;
        n = 0;
        room = kMax;
    }

    // want buffers of at least `bytes` each, or need of them where memory does not hold want: the number that may be
    // used, 0 when not even need fit (nothing is held then).  What is held is not given up for a number that may
    // not fit, and a number that did not fit is not asked for again while the set is held, so that a repeated call
    // allocates and frees nothing.
    template <class Alloc, class Free> int get(size_t bytes, int need, int want, Alloc alloc, Free release) {
        if (cap < bytes) {
            clear(release);
            cap = bytes;
        }
        const int before = n, target = want <= room ? want : need;
        while (n < target && (p[n] = alloc(cap))) ++n;
        if (n >= target) return target;
        if (n >= need) {
            room = n;
            while (n > need && n > before) release(p[--n]);
            p[n] = nullptr;
            return need;
        }
        const bool larger = cap > bytes;
        clear(release);
        return larger ? get(bytes, need, want, alloc, release) : 0;
    }
};

}  // namespace pa
