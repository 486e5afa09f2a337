// metric.hpp -- level metrics and other tables that no kernel writes, read
// through the constant address space.
#pragma once
#include <hip/hip_runtime.h>

namespace mimadv {

// A table of the context (metrics, coefficients).  Read at a wave-uniform index
// it takes a scalar load.  Through an ordinary pointer the compiler must
// assume that the kernel's stores may change it and uses a vector load, whose
// wait also drains every load the kernel has requested ahead of its use
// (measured with the vector loads and without, same bits: 48 uneven subdomains
// 15.35 -> 13.06 ms per step, 20 fields at 512x512x160 19.3 -> 18.4 ms, PPM
// 256 -> 242 us and 'weno' 158 -> 152 us per field at 256x256x128, four
// adjoint steps there 5.32 -> 5.10 ms).
template <class T>
using Table = const __attribute__((address_space(4))) T *;

template <class T>
__device__ __forceinline__ Table<T> table(const T *p)
{
    return (Table<T>)p;
}

}  // namespace mimadv
