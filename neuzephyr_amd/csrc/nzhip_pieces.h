// 16-byte pieces at 4-byte aligned addresses, for the kernels that read rows of any width and alignment.
#ifndef NZHIP_PIECES_H
#define NZHIP_PIECES_H

#include <hip/hip_runtime.h>

namespace nzhip {

typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float floatx2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float piece4 __attribute__((ext_vector_type(4)));

// element e of a piece that was moved back by `back` elements; what lies beyond the extent comes out as some element of it
__device__ __forceinline__ piece4 turn_back(const piece4 q, int back) {
    const float a = back & 1 ? q[1] : q[0], b = back & 1 ? q[2] : q[1], c = back & 1 ? q[3] : q[2];
    return piece4{back & 2 ? c : a, back & 2 ? q[3] : b, c, q[3]};
}

}  // namespace nzhip

#endif
