// Launch grids of the tracer kernels that take several threads per tracer
// (csrc/lpt_kernels.hpp: thread_grid, thread_at): for every count given, the threads
// along each axis below 2^32 (the runtime counts them in 32 bits) and blocks y below
// 2^16, every place below n taken once: consecutive blocks continue each other, the
// first starts at 0 and the last reaches n.  Exit status 1 otherwise.
#include <cstdio>
#include <cstdlib>

#include "lpt_kernels.hpp"

int main(int argc, char** argv)
{
    for (int k = 1; k < argc; k++) {
        const long n = std::atol(argv[k]);
        const dim3 g = lpt::thread_grid(n, 8);
        bool ok = (unsigned long)g.x * 256 < (1ul << 32) && g.y < 65536 && g.z == 8;
        ok = ok && lpt::thread_at(0, 0, 0) == 0 && lpt::thread_at(g.x - 1, g.y - 1, 255) >= n - 1;
        for (unsigned y = 0; y < g.y; y++) {
            ok = ok && lpt::thread_at(0, y, 255) == lpt::thread_at(0, y, 0) + 255;
            if (g.x > 1) ok = ok && lpt::thread_at(1, y, 0) == lpt::thread_at(0, y, 0) + 256;
            if (y) ok = ok && lpt::thread_at(0, y, 0) == lpt::thread_at(g.x - 1, y - 1, 255) + 1;
        }
        std::printf("%ld threads: %u x %u x %u blocks%s\n", n, g.x, g.y, g.z, ok ? "" : "  WRONG");
        if (!ok) return 1;
    }
    return 0;
}
