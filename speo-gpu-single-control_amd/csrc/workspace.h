// workspace.h -- a device buffer that grows to what its owner's calls need and is
// kept until the owner goes.
#pragma once

#include <cstddef>
#include <cstdint>

namespace speo {

struct Workspace {
    float *p = nullptr;
    size_t cap = 0;               // floats at p
    size_t refused = SIZE_MAX;    // the least the device has had no room for

    // At least `least` floats at p, `want` (>= least) where the device has room and
    // the call may allocate.  What is refused once is not asked for again where
    // the call can do without: a failed allocation costs more than it.  Mem:
    //   bool may_allocate()              false inside a stream capture
    //   int settle()                     waits for the buffer's users
    //   int allocate(float **, size_t)   0, kNoRoom or another error
    //   void release(float *)
    static constexpr int kNoRoom = -1;
    template <typename Mem> int reserve(size_t least, size_t want, Mem &mem) {
        if (want <= cap) return 0;
        if (least <= cap) {
            // the buffer does; a larger one replaces it only once it is there
            if (want >= refused || !mem.may_allocate()) return 0;
            float *q = nullptr;
            const int rc = mem.allocate(&q, want);
            if (rc == kNoRoom) {
                refused = want;
                return 0;
            }
            if (rc) return rc;
            if (const int e = cap ? mem.settle() : 0) {
                mem.release(q);
                return e;
            }
            mem.release(p);
            p = q;
            cap = want;
            return 0;
        }
        if (const int e = mem.settle()) return e;
        mem.release(p);
        p = nullptr;
        cap = 0;
        if (want < refused || want == least) {
            const int rc = mem.allocate(&p, want);
            if (rc == 0) cap = want;
            if (rc == kNoRoom && want < refused) refused = want;
            if (rc != kNoRoom || want == least) return rc;
        }
        const int rc = mem.allocate(&p, least);
        if (rc == 0) cap = least;
        return rc;
    }
};

}  // namespace speo
