// Host check of what a failed device allocation does: the handle of the running
// call gives its spare memory back once, then the allocation is tried again.
#include <cstdlib>
#include <thread>

#include "common.hpp"

static int fails = 0, tries = 0, given = 0;
extern "C" {
hipError_t hipMalloc(void** p, size_t)
{
    tries++;
    if (fails > 0) {
        fails--;
        return hipErrorOutOfMemory;
    }
    *p = std::malloc(16);
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "out of memory"; }
}

static void give(void* owner) { given += *static_cast<int*>(owner); }

// Result of one allocation: 1 done, 0 refused; tries and given count from 0.
static int one(int failing)
{
    fails = failing;
    tries = given = 0;
    regot::DBuf<double> b;
    try {
        b.alloc(5);
    } catch (const regot::Error& e) {
        return e.code == regot::E_NOMEM && b.p == nullptr && b.n == 0 ? 0 : -1;
    }
    return b.n == 5 ? 1 : -1;
}

#define CHECK(x)                                  \
    do {                                          \
        if (!(x)) {                               \
            std::printf("failed: %s\n", #x);      \
            return 1;                             \
        }                                         \
    } while (0)

int main()
{
    int ten = 10, one_ = 1;
    CHECK(one(0) == 1 && tries == 1);
    CHECK(one(1) == 0 && tries == 1);   // nothing to give back
    {
        regot::SpareScope outer(&ten, give);
        CHECK(one(0) == 1 && given == 0);
        CHECK(one(1) == 1 && tries == 2 && given == 10);
        CHECK(one(2) == 0 && tries == 2 && given == 10);
        {
            regot::SpareScope inner(&one_, give);
            CHECK(one(1) == 1 && given == 1);
        }
        CHECK(one(1) == 1 && given == 10);
        int other = -1;
        std::thread([&] { other = one(1); }).join();   // another thread's call
        CHECK(other == 0 && given == 0);
    }
    CHECK(one(1) == 0 && given == 0);
    return 0;
}
