// Host build of the wide tile kernel's row addresses (wide_core.h).  Input
// lines: <rows of the block> <waves> <rows that exist> <ld> <dim>.  Every load of
// every wave, lane, row piece and K stage is walked; per line it prints
//   <loads in range that leave the caller's rows> <elements the arithmetic needs
//   whose load is out of range> <offsets beyond 31 bits>
// and "refused" for strides the kernel does not take.  The caller's rows are
// (nrows - 1) ld + dim floats, in 16-byte groups.
#include <cstdint>
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>

#include "wide_core.h"

int main() {
    using namespace speo;
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        int rb, nw, nrows, ld, dim;
        in >> rb >> nw >> nrows >> ld >> dim;
        if (!wide_stride_fits(rb, ld)) {
            std::printf("refused\n");
            continue;
        }
        const int64_t owned = ((int64_t)(nrows - 1) * ld + round_up(dim, 4)) * 4, limit = wide_row_bytes(nrows, ld, dim);
        long outside = 0, needed = 0, wide = 0;
        for (int w = 0; w < nw; ++w)
            for (int lane = 0; lane < 64; ++lane)
                for (int j = 0; j < rb / 8 / nw; ++j)
                    for (int s = 0; s < (dim + 31) / 32; ++s) {
                        const int64_t scalar = (int64_t)j * 8 * nw * ld * 4 + 128 * s;
                        const int64_t at = wide_row_offset(w, lane, ld) + scalar;
                        const int row = 8 * (w + nw * j) + lane / 8;
                        const int64_t col = (at - (int64_t)row * ld * 4) / 4;
                        wide += at > 0x7fffffff || scalar > 0x7fffffff || limit > 0x7fffffff || limit < 0;
                        const bool read = at + 16 <= limit;
                        outside += read && at + 16 > owned;
                        needed += !read && row < nrows && col >= 0 && col < dim;
                    }
        std::printf("%ld %ld %ld\n", outside, needed, wide);
    }
    return 0;
}
