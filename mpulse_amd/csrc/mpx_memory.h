// Device memory: allocation, and the one block per GPU kept between adjoint calls (mpx_memory.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace mpx {

// hipMalloc; out of memory frees the kept blocks, if there are any, and tries once more
hipError_t dev_malloc(void **p, size_t bytes);
template <typename T>
hipError_t dev_malloc(T **p, size_t bytes)
{
    return dev_malloc((void **)p, bytes);
}

// frees the kept blocks; whether there was one
bool spare_drop();
// a block of at least *bytes (its size returned), the kept one if it is large enough; null on failure
void *spare_take(int device, size_t *bytes);
// puts a block back that no kernel uses any more; the slot's older block, or this one past the bound
// or with no solver alive, is freed
void spare_give(int device, void *p, size_t bytes);
// a solver is made (+1) or destroyed (-1); the last one takes the kept blocks with it
void spare_solvers(int change);

}  // namespace mpx
