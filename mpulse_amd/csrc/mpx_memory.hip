// An adjoint call works in gigabytes that it needs for its own length only.  Allocating and
// freeing them on every call took 60 (250 separate arrays) to 90 ms (one block: the driver clears
// what it maps) of the 157 ms of a 128x128x256, 100-step gradient, so one block per GPU is kept
// between calls, whichever solver they are for.  It holds nothing: a call takes the block out of
// its slot (a second call at the same time finds the slot empty and allocates), uses it on its own
// stream and puts it back after waiting for that stream.  Bounded to an eighth of the GPU's
// memory; freed by mpx_release_memory, with the last solver, and when an allocation of this library
// (hipFFT's plans included) finds the GPU full, which is then tried again.
#include "mpx_memory.h"

#include <mutex>
#include <utility>
#include <vector>

namespace mpx {

namespace {
struct Spare {
    void *p = nullptr;
    size_t bytes = 0;
};
std::mutex g_mu;
std::vector<Spare> g_spare;  // per device id
int g_solvers = 0;           // solvers alive
}  // namespace

bool spare_drop()
{
    std::vector<Spare> old;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        old.swap(g_spare);
    }
    bool any = false;
    for (const Spare &b : old)
        if (b.p) any = hipFree(b.p) == hipSuccess || any;
    return any;
}

hipError_t dev_malloc(void **p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory && spare_drop()) {
        (void)hipGetLastError();
        e = hipMalloc(p, bytes);
    }
    return e;
}

void *spare_take(int device, size_t *bytes)
{
    Spare b;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (device < (int)g_spare.size()) std::swap(b, g_spare[device]);
    }
    if (b.p && b.bytes >= *bytes) {
        *bytes = b.bytes;
        return b.p;
    }
    if (b.p) (void)hipFree(b.p);
    void *p = nullptr;
    if (dev_malloc(&p, *bytes) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return p;
}

void spare_give(int device, void *p, size_t bytes)
{
    if (!p) return;
    size_t avail = 0, total = 0;
    Spare b{p, bytes};
    if (hipMemGetInfo(&avail, &total) == hipSuccess && bytes <= total / 8) {
        std::lock_guard<std::mutex> lock(g_mu);
        if (g_solvers > 0) {
            if ((int)g_spare.size() <= device) g_spare.resize(device + 1);
            std::swap(b, g_spare[device]);
        }
    }
    if (b.p) (void)hipFree(b.p);
}

void spare_solvers(int change)
{
    bool last;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        g_solvers += change;
        last = g_solvers == 0;
    }
    if (last) (void)spare_drop();
}

}  // namespace mpx
