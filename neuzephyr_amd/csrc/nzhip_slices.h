// Pieces of the kernels whose waves cut the contraction of one output tile between them (nzhip_gemm_slices.hip, nzhip_conv_slices.hip).
#ifndef NZHIP_SLICES_H
#define NZHIP_SLICES_H

#include <hip/hip_runtime.h>

#include "nzhip_lds_tiles.h"
#include "nzhip_pieces.h"

namespace nzhip {

typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
constexpr int SLICE_PITCH = 80;                                      // bytes of an LDS row of 32 halfs: 16-byte reads of 32 rows meet no bank twice

__device__ __forceinline__ __amdgpu_buffer_rsrc_t slice_buffer(const float* x, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), 0, bytes, CL_RSRC);
}
// what a lane of this wave wrote to LDS is there for the others, and what they still read is not overwritten
__device__ __forceinline__ void slice_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// A wave's sums into LDS, four rows of a column at a time: unit (i, g, j) holds rows 8 g + 4 (lane >> 5) .. + 3 of block (i, j)
template <int FM, int FN>
__device__ __forceinline__ void slice_park(piece4* park, const floatx16 (&acc)[FM][FN], int wave, int lane) {
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                park[((wave * FM * 4 + i * 4 + g) * FN + j) * 64 + lane] = piece4{acc[i][j][g * 4], acc[i][j][g * 4 + 1], acc[i][j][g * 4 + 2], acc[i][j][g * 4 + 3]};
}
// the sum of the `active` waves' unit, added in pairs
template <int FM, int FN, int NW>
__device__ __forceinline__ piece4 slice_collect(const piece4* park, int ig, int j, int active, int lane) {
    piece4 o[NW];                                                   // all requested before the first is added
#pragma unroll
    for (int w = 0; w < NW; w++) o[w] = park[(((w < active ? w : 0) * FM * 4 + ig) * FN + j) * 64 + lane];
#pragma unroll
    for (int w = 1; w < NW; w++)
#pragma unroll
        for (int e = 0; e < 4; e++) o[w][e] = w < active ? o[w][e] : 0.f;
#pragma unroll
    for (int h = NW / 2; h > 0; h /= 2)
#pragma unroll
        for (int w = 0; w < h; w++)
#pragma unroll
            for (int e = 0; e < 4; e++) o[w][e] += o[w + h][e];
    return o[0];
}

}  // namespace nzhip

#endif
