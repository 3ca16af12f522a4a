/*
 * publish_device.cuh -- the store of a value that another block of the same launch reads (the site fronts). The card's dies
 * have a level-2 cache each, and a plain store stays in its own die's: a block of another die would read what was there before.
 * A relaxed store of agent scope goes through that cache. Every value that is published is stored here, as the publication
 * itself (front_publish) waits for the stores and writes nothing back.
 */
#ifndef PUBLISH_DEVICE_CUH
#define PUBLISH_DEVICE_CUH

#include <hip/hip_runtime.h>

template <typename T> __device__ static __forceinline__ void store_through(T *to, T value)
{
    static_assert(sizeof(T) == 4u || sizeof(T) == 8u, "one store of a lane");
    __hip_atomic_store(to, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

#endif
