// Host build of the growing workspace (workspace.h) over a made-up device of
// <room> floats.  Input lines: "R <least> <want> <may allocate>" (one reserve), "M <room>".
// Output per R: <status> <floats held> <allocations tried> <waits> <live buffers>.
#include <cstdio>
#include <cstdlib>
#include <iostream>
#include <map>
#include <sstream>
#include <string>

#include "workspace.h"

struct Device {
    size_t room = 0, used = 0;
    bool may = true;
    int tried = 0, waits = 0;
    std::map<float *, size_t> live;
    bool may_allocate() { return may; }
    int settle() { return ++waits, may ? 0 : 7; }  // a wait is an error inside a capture
    int allocate(float **out, size_t n) {
        ++tried;
        if (used + n > room) return speo::Workspace::kNoRoom;
        *out = static_cast<float *>(std::malloc(1));
        live[*out] = n;
        used += n;
        return 0;
    }
    void release(float *p) {
        if (!p) return;
        used -= live.at(p);
        live.erase(p);
        std::free(p);
    }
};

int main() {
    Device dev;
    speo::Workspace w;
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        char kind;
        in >> kind;
        if (kind == 'M') {
            in >> dev.room;
            continue;
        }
        size_t least, want;
        int may;
        in >> least >> want >> may;
        dev.may = may != 0;
        dev.tried = dev.waits = 0;
        const int rc = w.reserve(least, want, dev);
        if ((w.cap != 0) != (w.p != nullptr) || (w.p && dev.live.at(w.p) != w.cap)) return 1;
        std::printf("%d %zu %d %d %zu\n", rc, w.cap, dev.tried, dev.waits, dev.live.size());
    }
    return 0;
}
