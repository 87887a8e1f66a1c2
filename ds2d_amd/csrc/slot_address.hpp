// Addresses in a window for the kernels whose waves hold one column each.
#pragma once
#include <cstdint>

namespace ds2d {

// Element where column ix of a window at element off starts, columns of nz
// elements.  Uniform over a wave: 64 bits in scalar registers.
__host__ __device__ inline long long column_start(long long off, int ix, int nz) { return off + (long long)ix * nz; }

// Element z of the column of f that starts at element start: a lane adds 32
// bits of byte offset within its column, so that windows may have any number
// of cells and an access still costs no 64-bit vector arithmetic.
template <typename T>
__host__ __device__ inline T& column_cell(T* f, long long start, int z) {
    const char* column = reinterpret_cast<const char*>(f + start);
    return *const_cast<T*>(reinterpret_cast<const T*>(column + (uint32_t)z * (uint32_t)sizeof(T)));
}

}  // namespace ds2d
