// Error bits raised by kernels: one word per bit in pinned host memory that
// the kernels store to and the host reads after it has waited for the
// stream, so a synchronous call needs no copy.  Plain stores, each bit in
// its own word: no atomic goes over the bus, and nothing is written at all
// unless an error is found.
#pragma once

#include <hip/hip_runtime.h>

namespace ucfd {

// raise one UCFD_KFLAG_* bit (no cross-lane step: one in the sweep kernels'
// face loops cost them 3 % through the order of their loads)
__device__ __forceinline__ void raise(int *words, int bit)
{
    __hip_atomic_store(words + __builtin_ctz(bit), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace ucfd
