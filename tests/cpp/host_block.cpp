// The end of a pinned block (reg.hpp, HostBlock) when the host is out of
// memory: the block is given back and the call goes on.  The HIP runtime's
// calls and operator new are this program's own.
#include <cstdio>
#include <cstdlib>
#include <new>

#include "../../qvnt_amd/csrc/reg.hpp"

static bool out_of_memory = false;
static int allocated = 0, freed = 0;

void* operator new(std::size_t n) {
    if (out_of_memory) throw std::bad_alloc();
    void* p = std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

extern "C" hipError_t hipHostMalloc(void** p, size_t n, unsigned int) {
    ++allocated;
    *p = std::malloc(n);
    return hipSuccess;
}
extern "C" hipError_t hipHostFree(void* p) {
    ++freed;
    std::free(p);
    return hipSuccess;
}
extern "C" hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}

#define CHECK(x) if (!(x)) { std::printf("failed: %s\n", #x); return 1; }

int main() {
    void* kept = nullptr;
    {
        qvnt::HostBlock b(0, 4096);
        CHECK(b.p && allocated == 1);
        kept = b.p;
    }
    CHECK(freed == 0);
    {
        qvnt::HostBlock b(0, 4096);   // the block kept
        CHECK(b.p == kept && allocated == 1);
        out_of_memory = true;
    }
    out_of_memory = false;
    CHECK(freed == 1);                // there was no memory to remember it in
    {
        qvnt::HostBlock b(0, 4096);
        CHECK(b.p && allocated == 2);
    }
    CHECK(freed == 1);
    std::puts("ok");
    return 0;
}
