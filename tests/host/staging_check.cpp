// Host check of the pinned staging memory's size: the HIP runtime's allocation
// calls are replaced by ones that record the bytes asked for.
#include <cstdlib>

#include "problem.hpp"

static size_t asked = 0;
extern "C" {
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned int)
{
    asked = bytes;
    *p = std::malloc(64);   // never touched beyond its first entries
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned int)
{
    *d = h;
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return ""; }
}

int main()
{
    const int sizes[][2] = {{1, 1}, {16384, 16384}, {1, (1 << 30) - 1}, {1, 1 << 30},
                            {1100000000, 1}, {1 << 30, (1 << 30) - 1}};
    for (const auto& q : sizes) {
        const size_t nm = static_cast<size_t>(q[0]) + static_cast<size_t>(q[1]);
        regot::MappedRing<double> ring;
        ring.ensure(regot_problem::stage_size(q[0], q[1]));
        const size_t in = regot_problem::kStageAt, out = regot_problem::stage_out_at(q[0], q[1]);
        // scalars, then n + m values in, then n + m values out
        if (out < in + nm || asked != 8 * (64 + 2 * nm) || ring.cap * 8 != asked ||
            out + nm > ring.cap) {
            std::printf("%d x %d: %zu bytes, out at %zu\n", q[0], q[1], asked, out);
            return 1;
        }
    }
    std::puts("staging sizes ok");
    return 0;
}
