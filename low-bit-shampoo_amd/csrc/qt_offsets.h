// Byte offsets into one quantized square matrix.  order * order stays below 2^31 (checked on the host), so the index of an
// element fits an int and the offset of its code 32 bits -- but not the index times the bits of a code, which passes 2^31
// from order 16384 (8 bits) and 23171 (4 bits) on.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#define QT_EITHER_SIDE __host__ __device__ __forceinline__
#else
#define QT_EITHER_SIDE inline
#endif

namespace qt {

// of the code of element (row, col); 4 bits: of the byte that holds it
template <int BITS>
QT_EITHER_SIDE uint32_t code_offset(int row, int col, int order) {
    const uint32_t element = (uint32_t)(row * order + col);
    return BITS == 4 ? element >> 1 : element;
}

// of a row's first segment maximum
QT_EITHER_SIDE uint32_t absmax_offset(int row, int order, int bs_shift) { return (uint32_t)(row * (order >> bs_shift)) * 4u; }

}  // namespace qt
