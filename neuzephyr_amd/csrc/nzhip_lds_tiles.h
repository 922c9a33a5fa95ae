// Pieces of the kernels that stream fp16 copies of their operands into LDS (nzhip_conv_cl.hip, nzhip_gemm_copy.hip).
#ifndef NZHIP_LDS_TILES_H
#define NZHIP_LDS_TILES_H

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nzhip {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

static int round8(int c) { return (c + 7) / 8 * 8; }
// Elements from one row of a copy to the next, for rows of n: an odd number of 128-byte lines. A tile loads the same lines of 64 rows at
// once, and the channels of a level-2 cache take 256 bytes in turn: rows an even number of lines apart crowd on half of them and fewer.
static int cl_pitch(int n) {
    const int lines = (n + 63) / 64;
    return n <= 64 ? round8(n) : (lines | 1) * 64;
}

constexpr unsigned CL_RSRC = 0x00020000;                            // raw buffer, offsets in bytes, zeros past num_records
constexpr unsigned CL_OUT = 0x80000000u;                            // an offset past any of the copies (all below 2 GiB)

template <int N>
__device__ __forceinline__ void cl_wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0070 | 0x0F00);
}
// 16 bytes a lane from r + off to LDS address `lds` + 16 lane, zeros where off is past the buffer's end. In assembly because the compiler
// would have every LDS read after it wait for all requests in flight; it has no register output, and the kernels wait by count.
typedef int int4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int4_t cl_buffer(const void* base, unsigned bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return int4_t{(int)(uint32_t)a, (int)(uint32_t)(a >> 32), (int)bytes, (int)CL_RSRC};
}
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"                   // m0 is reserved: that it is not preserved across the assembly is what is said here
__device__ __forceinline__ void cl_load(int4_t r, unsigned lds, unsigned off) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(r), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ unsigned cl_lds(const char* p) { return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const char*)p; }
// n / d for n below 2^31: one product and a shift (a division by a run-time value is some 40 instructions, and a workgroup needs a
// dozen of them before its first request)
struct ClDiv {
    unsigned m;
    int sh;
};
static ClDiv cl_div(unsigned d) {
    int l = 0;
    while ((1ull << l) < d) l++;
    return ClDiv{(unsigned)((1ull << (31 + l)) / d + (((1ull << (31 + l)) % d) != 0)), 31 + l};
}
__device__ __forceinline__ int cl_quot(int n, ClDiv d) { return (int)(((unsigned long long)(unsigned)n * d.m) >> d.sh); }
// workgroup -> place in a list, so that every XCD (workgroups go to them round-robin) walks one contiguous stretch of it
__device__ __forceinline__ int cl_xcd_place(int lin, int total) {
    const int xcd = lin & 7, q = lin >> 3, per = total >> 3, rem = total & 7;
    return xcd * per + (xcd < rem ? xcd : rem) + q;
}
// the 8 contraction elements of this lane's fragment row from two halves of LDS rows that hold one contraction element each: 16 lanes
// read 4 rows x 16 columns, lane i gets column i of the 4 rows
__device__ __forceinline__ half8_t cl_read_turned(const char* lo, const char* hi) {
    const short4_t l = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)lo);
    const short4_t h = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)hi);
    const half4_t a = __builtin_bit_cast(half4_t, l), b = __builtin_bit_cast(half4_t, h);
    half8_t v;
#pragma unroll
    for (int e = 0; e < 4; e++) { v[e] = a[e]; v[4 + e] = b[e]; }
    return v;
}

// Sums of the steps so far, which a chain leaves after every `chain` of them: the error of an fp32 sum grows with the length of its chain,
// and the kernels these take the place of cut a long contraction into chunks. Products: chains of CL_CHAIN steps, 512 elements. 944 x 2352 x 1984
// has a relative error of 1.5e-7 against 64 bits then, 3.1e-7 without, 2.2e-7 on the fused kernel. It costs 1 to 2 %
// (1000 x 777 x 513 11.3 -> 11.5 us, both gradients of 4096 x 1024 -> 4096 112 -> 115).
constexpr int CL_CHAIN = 8;
// Convolutions and products of at most 64 rows or columns: the kernels before sum in chunks of 16 channels, 128 pixels, 128 elements. n steps a chain of S leave an error of about 8.7 n + S / n
// squared (fitted to chains of 1, 2, 4 and 8 steps), least at these n. Chains of 512 were up to 1.8 times as far off as those kernels
// (weight gradient 8 x 13 x 16 x 16 -> 128, 7x7 at stride 2 1.4e-7, 0.8e-7 before and now). They cost 1 % more than those.
__host__ __device__ __forceinline__ int cl_chain(int steps) { return steps < 18 ? 1 : steps < 70 ? 2 : steps < 280 ? 4 : steps < 1120 ? 8 : 16; }
// The parts' sums, eight chains side by side for the same reason (64 in one chain: 1.6e-7, weight gradient 4 x 16 x 32 x 32 -> 16, 1.0e-7 so)
template <typename F>
__device__ __forceinline__ float cl_sum_parts(int parts, F part) {
    float s[8] = {};
    for (int q = 0; q < parts; q += 8) {                              // all eight requested before the first is added
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = part(q + e < parts ? q + e : parts - 1);
#pragma unroll
        for (int e = 0; e < 8; e++) s[e] += q + e < parts ? v[e] : 0.f;
    }
    return ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));
}
template <int TM, int TN>
struct ClSums {
    floatx16 sum[TM][TN];
    __device__ __forceinline__ ClSums() {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) sum[i][j][r] = 0.f;
    }
    // before the MFMAs of a step, between the requests of its fragments and their use: the time these take covers it. chain: a power of two
    __device__ __forceinline__ void take(floatx16 (&acc)[TM][TN], int step, int chain) {
        if (step & (chain - 1)) return;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    sum[i][j][r] += acc[i][j][r];
                    acc[i][j][r] = 0.f;
                }
    }
    __device__ __forceinline__ void finish(floatx16 (&acc)[TM][TN]) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += sum[i][j][r];
    }
};

// The kernels ask for two waves per SIMD, the most that LDS has room for: with up to 256 registers the compiler keeps the sums in ordinary ones, with
// up to 512 in accumulation registers, and every sum that a chain leaves would be moved there and back.
// A tile: TM x TN fragments of 32 x 32 per wave, 2 x WN waves in each of KG groups.
template <int TM_, int TN_, int WN_, int KG_>
struct ClTile {
    static constexpr int TM = TM_, TN = TN_, WN = WN_, KG = KG_;
    static constexpr int BM = 64 * TM, BN = 32 * TN * WN, GROUP = 128 * WN, THREADS = GROUP * KG;
    static constexpr int STAGE = (BM + BN) * 128, NST = BM + BN == 192 || BM + BN > 256 ? 3 : 4, RING = KG * NST * STAGE;
    static constexpr int LA = BM / 16 / WN, LB = BN / 16 / WN;       // requests of 8 rows per wave and step
};

}  // namespace nzhip

#endif
