// Products on rounded copies: one launch rounds the operands to fp16 as they lie (rows of contiguous elements, LDS-friendly pitch), a second
// one multiplies the copies, for one product or for two that share an operand (both gradients of a Linear layer).
//
// The fused kernel rounds every fp32 tile where it stages it, through registers: a CU takes tiles in at 50 GB/s that way, and every
// operand element is rounded once per tile that uses it. From the copies tiles go to LDS without registers at half the bytes
// (nzhip_lds_tiles.h). Unlike the block images of the two-pass route (nzhip_gemm_h16.hip) the copies keep the operand's own layout:
// an operand whose contraction runs along its rows is read in 16-byte pieces of the contraction, one whose contraction runs across
// them through the transposing LDS load, so one copy serves both products and rounding is a plain stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "nzhip_internal.h"
#include "nzhip_lds_tiles.h"
#include "nzhip_pieces.h"
#include "nzhip_plan_cache.h"

namespace nzhip {

// ---- the copies ------------------------------------------------------------------------------------------------
struct CopyJob {
    const float* src;
    _Float16* dst;
    long ld;                            // of src
    int rows, cols, pitch, blocks;
    ClDiv by_units;                     // units of 8 elements per row
};
struct CopyJobs { CopyJob job[4]; };

// Bound by memory: 16 MB of fp32 to 8 MB of fp16 in 5 us. A thread takes 8 elements, 32 bytes in and 16 out; elements past a row's end are zeros.
__global__ __launch_bounds__(256) void round_rows_kernel(const CopyJobs a) {
    int b = blockIdx.x, n = 0;
    while (n < 3 && b >= a.job[n].blocks) b -= a.job[n++].blocks;
    const CopyJob& j = a.job[n];
    const int units = (j.cols + 7) / 8, u = b * 256 + threadIdx.x, row = cl_quot(u, j.by_units), c = (u - row * units) * 8;
    if (row >= j.rows) return;
    const float* s = j.src + row * j.ld + c;
    half8_t h;
    if (c + 8 <= j.cols) {
        const piece4 lo = *reinterpret_cast<const floatx4u*>(s), hi = *reinterpret_cast<const floatx4u*>(s + 4);
#pragma unroll
        for (int e = 0; e < 4; e++) { h[e] = (_Float16)lo[e]; h[4 + e] = (_Float16)hi[e]; }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = c + e < j.cols ? (_Float16)s[e] : (_Float16)0.f;
    }
    *reinterpret_cast<half8_t*>(j.dst + (long)row * j.pitch + c) = h;
}

// ---- the product ---------------------------------------------------------------------------------------------------
struct CopyProduct {
    const _Float16* A;                  // A_KC: M rows along k, else K rows along m
    const _Float16* B;                  // B_KC: N rows along k, else K rows along n
    float* C;
    const float* bias;
    float* partial;                     // [part][M][N] bare sums, or null
    int M, N, K, lda, ldb, ldc;
    unsigned a_bytes, b_bytes;
    long bias_sm, bias_sn;
    int relu, parts, part_steps, tiles, tiles_m, tiles_n, chain;      // chain: steps, a power of two
    ClDiv by_tiles, by_panel;           // panels of up to 8 tile columns
};
struct CopyPair {
    CopyProduct p[2];
    int total, head;                    // workgroups; those of the product with the longer sums, which start first
    int longer;                         // that product
};

// One workgroup tile of one product; lin: its place in the product's list of (part, tile). LDS rows and swizzle as in the convolution
// kernels: an operand along k has rows of 64 k, one across k has 64 rows of k, 64 columns each, per 64 columns of the tile.
// Rows, columns and k past the end come out of the buffers' bounds as zeros, k past the end of a row by a test per request.
template <bool A_KC, bool B_KC, typename T>
__device__ __forceinline__ void copy_tile(const CopyProduct& p, const int lin, char* lds) {
    constexpr int TM = T::TM, TN = T::TN, KG = T::KG, BM = T::BM, BN = T::BN, NST = T::NST, STAGE = T::STAGE;
    constexpr int LA = T::LA, LB = T::LB, LOADS = LA + LB, Q = 4 / T::WN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & (2 * T::WN - 1), kg = KG > 1 ? __builtin_amdgcn_readfirstlane(tid / T::GROUP) : 0;
    const int wm = wave / T::WN, wn = wave % T::WN, li = lane & 31, lh = lane >> 5;

    const int part = cl_quot(lin, p.by_tiles), t = lin - part * p.tiles;
    const int panel = cl_quot(t, p.by_panel), wide = p.tiles_n - panel * 8 < 8 ? p.tiles_n - panel * 8 : 8, in = t - panel * 8 * p.tiles_m;
    const int tile_m = wide == 8 ? in >> 3 : in / wide, tile_n = panel * 8 + in - tile_m * wide;
    const int m0 = tile_m * BM, n0 = tile_n * BN;

    const int all = (p.K + 63) / 64, step0 = part * p.part_steps, last = step0 + p.part_steps < all ? step0 + p.part_steps : all;
    const int steps = (last - step0 + KG - 1) / KG, units = last == all ? (p.K + 7) / 8 : last * 8;
    const int4_t ra = cl_buffer(p.A, p.a_bytes), rb = cl_buffer(p.B, p.b_bytes);

    // this lane's slot in a group of 8 LDS rows holds unit ch of the row in even groups, ch ^ 4 in odd ones
    const int ch = (lane & 7) ^ (lane >> 4);
    unsigned off_a[LA], off_b[LB];
    auto start = [&](unsigned* off, bool kc, int count, int first, int ld) {
#pragma unroll
        for (int j = 0; j < (LA > LB ? LA : LB); j++) {
            if (j >= count) break;
            if (kc) off[j] = (unsigned)((first + (wave * count + j) * 8 + (lane >> 3)) * ld + (step0 + kg) * 64 + (ch ^ ((j & 1) * 4)) * 8) * 2u;
            else {
                const int g = wave * Q + j % Q;
                off[j] = (unsigned)(((step0 + kg) * 64 + g * 8 + (lane >> 3)) * ld + first + (j / Q) * 64 + (ch ^ ((g & 1) * 4)) * 8) * 2u;
            }
        }
    };
    start(off_a, A_KC, LA, m0, p.lda);
    start(off_b, B_KC, LB, n0, p.ldb);
    const unsigned add_a = (A_KC ? 64u : 64u * (unsigned)p.lda) * 2u * KG, add_b = (B_KC ? 64u : 64u * (unsigned)p.ldb) * 2u * KG;
    int at = (step0 + kg) * 8;                                      // first unit of the next request's step

    char* ring = lds + kg * NST * STAGE;
    const unsigned at_a = cl_lds(ring) + wave * (A_KC ? LA : Q) * 1024, at_b = cl_lds(ring) + BM * 128 + wave * (B_KC ? LB : Q) * 1024;
    auto request_one = [&](int slot, int j) {                       // the step's j-th request
        if (j < LA) {
            const unsigned to = at_a + slot * STAGE + (A_KC ? j * 1024 : (j / Q) * 8192 + (j % Q) * 1024);
            cl_load(ra, to, at + (A_KC ? ch ^ ((j & 1) * 4) : 0) < units ? off_a[j] : CL_OUT);
            off_a[j] += add_a;
        } else {
            const int i = j - LA;
            const unsigned to = at_b + slot * STAGE + (B_KC ? i * 1024 : (i / Q) * 8192 + (i % Q) * 1024);
            cl_load(rb, to, at + (B_KC ? ch ^ ((i & 1) * 4) : 0) < units ? off_b[i] : CL_OUT);
            off_b[i] += add_b;
        }
        if (j == LOADS - 1) at += 8 * KG;
    };
    auto request = [&](int slot) {
#pragma unroll
        for (int j = 0; j < LOADS; j++) request_one(slot, j);
    };

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    // fragments: along k one 16-byte read; across k two transposing reads (16 lanes: 4 k x 16 columns)
    const int sw = (li >> 1) & 7, g = lane >> 4, i4 = lane & 15;
    int turned[2][2];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int f = 0; f < 2; f++) {
            const int r = (g >> 1) * 8 + h * 4 + (i4 >> 2), c = f * 4 + (g & 1) * 2 + ((i4 & 3) >> 1);
            turned[h][f] = r * 128 + ((c ^ ((r >> 1) & 7)) << 4) + (i4 & 1) * 8;
        }
    auto read = [&](const char* base, bool kc, int block, int k) {  // block: 32 rows or columns of the operand's tile
        if (kc) return *reinterpret_cast<const half8_t*>(base + (block * 32 + li) * 128 + ((((k << 1) | lh) ^ sw) << 4));
        const char* q = base + (block >> 1) * 8192 + k * 2048;
        return cl_read_turned(q + turned[0][block & 1], q + turned[1][block & 1]);
    };

    ClSums<TM, TN> sums;
    half8_t af[4][TM], bf[4][TN];
    auto fragments = [&](const char* base) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
#pragma unroll
            for (int i = 0; i < TM; i++) af[k][i] = read(base, A_KC, wm * TM + i, k);
#pragma unroll
            for (int j = 0; j < TN; j++) bf[k][j] = read(base + BM * 128, B_KC, wn * TN + j, k);
            __builtin_amdgcn_sched_barrier(0);                      // in the order of their use
        }
    };
    auto multiply = [&](int k) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[k][i], bf[k][j], acc[i][j], 0, 0, 0);
    };
    for (int s = 0; s < NST - 1; s++) request(s);
    int slot = 0;
    // 128 x 256: the waves of rows 0..63 and those of rows 64..127, one of each per SIMD, take turns: one half reads a step's fragments from LDS
    // while the other's MFMAs run and issue its requests, a barrier between the turns. All in step, the three added up (2560 clocks a
    // step of the pair below, of which the MFMAs are 1024, the reads about 900 and the issue of the requests 770): pairs of 4096 x 1024 -> 4096 116
    // -> 110 us, 4096 x 4096 -> 1024 130 -> 124, 2048^3 on this tile 45 -> 42. Left over is that either half alone takes 67 of the 87 us: with
    // the MFMAs out, with the requests out of bounds. Smaller tiles lose by the second barrier (2048^3 on 128 x 128 35.1 -> 36.6).
    // Half h of a step's two: the first half of the waves reads step s in half 2 s, the second in 2 s + 1, and each waits for its share of step s + 1
    // before the barrier that ends half 2 s + 1. A slot is free when the later half has read it: the first half fills the slot
    // of step s - 1 in half 2 s + 1, the second that of step s in half 2 s + 2, one step further ahead.
    if constexpr (TM == 2 && TN == 2) {
        static_assert(KG == 1 && T::WN == 4, "the halves are the waves of the tile's upper and lower rows, on the same SIMDs");
        const bool late = __builtin_amdgcn_readfirstlane(tid) >= T::THREADS / 2;
        cl_wait_vmcnt<(NST - 2) * LOADS>();
        if (late) {
            request(NST - 1);
            asm volatile("s_barrier" ::: "memory");
        }
        asm volatile("s_barrier" ::: "memory");
        for (int s = 0; s < steps; s++) {
            const int to = late ? slot : slot == 0 ? NST - 1 : slot - 1;
            fragments(ring + slot * STAGE);
            sums.take(acc, s, p.chain);
            __builtin_amdgcn_sched_barrier(0);
            if (late) cl_wait_vmcnt<(NST - 2) * LOADS>();
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                multiply(k);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = k * LOADS / 4; j < (k + 1) * LOADS / 4; j++) request_one(to, j);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
            if (!late) cl_wait_vmcnt<(NST - 2) * LOADS>();
            asm volatile("s_barrier" ::: "memory");
            slot = slot == NST - 1 ? 0 : slot + 1;
        }
        if (!late) asm volatile("s_barrier" ::: "memory");
    } else {
        for (int s = 0; s < steps; s++) {
            cl_wait_vmcnt<(NST - 2) * LOADS>();
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            request(slot == 0 ? NST - 1 : slot - 1);
            fragments(ring + slot * STAGE);
            sums.take(acc, s, p.chain);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 4; k++) multiply(k);
            __builtin_amdgcn_sched_barrier(0);
            slot = slot == NST - 1 ? 0 : slot + 1;
        }
    }
    sums.finish(acc);
    cl_wait_vmcnt<0>();

    if constexpr (KG > 1) {
        __syncthreads();
        floatx16* park = reinterpret_cast<floatx16*>(lds) + (wave * TM * TN) * 64 + lane;
        if (kg == 1) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) park[(i * TN + j) * 64] = acc[i][j];
        }
        __syncthreads();
        if (kg == 1) return;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const floatx16 o = park[(i * TN + j) * 64];
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += o[r];
            }
    }

    // lane = column, registers = rows (r >> 2) * 8 + lh * 4 + (r & 3); a tile's bias is read whole before its first store (it may be C)
    const bool split = p.parts > 1;
    const int ldo = split ? p.N : p.ldc;
    float* out = (split ? p.partial + (long)part * p.M * p.N : p.C) + (long)m0 * ldo;
    const float* bias = p.bias && !split ? p.bias + m0 * p.bias_sm : nullptr;
    if (bias) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = n0 + (wn * TN + j) * 32 + li, nc = n < p.N ? n : p.N - 1;
            if (p.bias_sm == 0) {
                const float v = bias[nc * p.bias_sn];
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[i][j][r] += v;
            } else {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int m = (wm * TM + i) * 32 + (r >> 2) * 8 + lh * 4 + (r & 3);
                        acc[i][j][r] += bias[(m0 + m < p.M ? m : 0) * p.bias_sm + nc * p.bias_sn];
                    }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = n0 + (wn * TN + j) * 32 + li;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = (wm * TM + i) * 32 + (r >> 2) * 8 + lh * 4 + (r & 3);
                float v = acc[i][j][r];
                if (p.relu && !split) v = v > 0.f ? v : 0.f;
                if (n < p.N && m0 + m < p.M) out[(unsigned)(m * ldo + n)] = v;
            }
    }
}

// FORM: bit 0 A_KC, bit 1 B_KC
template <int FORM, typename T>
__global__ __launch_bounds__(T::THREADS, 2) void copy_product_kernel(const CopyPair a) {
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    copy_tile<(FORM & 1) != 0, (FORM & 2) != 0, T>(a.p[0], cl_xcd_place(blockIdx.x, a.total), lds);
}
// Both gradients of C = A B: dA += dC B^T with dC along its rows, and dB += A^T dC across them. Each product's tiles are spread over all XCDs: their
// sums differ in length (rows of dC or columns), and in one list for both an XCD's stretch was of one product alone, the long
// sums on one or two XCDs of eight (1024 samples, 4096 inputs and outputs 219 -> 119 us, 8192 samples 943 -> 690).
template <int FORM1, int FORM2, typename T>
__global__ __launch_bounds__(T::THREADS, 2) void copy_pair_kernel(const CopyPair a) {
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int b = blockIdx.x;
    const bool tail = b >= a.head;
    const int lin = tail ? cl_xcd_place(b - a.head, a.total - a.head) : cl_xcd_place(b, a.head);
    if (tail == (a.longer == 1)) copy_tile<(FORM1 & 1) != 0, (FORM1 & 2) != 0, T>(a.p[0], lin, lds);
    else copy_tile<(FORM2 & 1) != 0, (FORM2 & 2) != 0, T>(a.p[1], lin, lds);
}

// C = act(the parts' sums + bias)
__global__ __launch_bounds__(256) void copy_sum_kernel(const CopyPair a, const int blocks1, const ClDiv by_n1, const ClDiv by_n2) {
    const bool second = (int)blockIdx.x >= blocks1;
    const CopyProduct& p = a.p[second];
    const int i = ((int)blockIdx.x - (second ? blocks1 : 0)) * 256 + threadIdx.x;
    if (i >= p.M * p.N) return;
    float s = cl_sum_parts(p.parts, [&](int q) { return p.partial[(long)q * p.M * p.N + i]; });
    const int m = cl_quot(i, second ? by_n2 : by_n1), n = i - m * p.N;
    if (p.bias) s += p.bias[m * p.bias_sm + n * p.bias_sn];
    if (p.relu) s = s > 0.f ? s : 0.f;
    p.C[(long)m * p.ldc + n] = s;
}

// ---- host side ----------------------------------------------------------------------------------------------------------
struct CopyShape { int bm, bn, kg; };
constexpr int COPY_TILES = 6;
constexpr CopyShape COPY_SHAPES[COPY_TILES] = {{64, 64, 1}, {64, 64, 2}, {128, 64, 1}, {64, 128, 1}, {128, 128, 1}, {128, 256, 1}};
template <typename F>
static int copy_pick(int tile, F go) {
    switch (tile) {
        case 0: return go(ClTile<1, 1, 2, 1>{});
        case 1: return go(ClTile<1, 1, 2, 2>{});
        case 2: return go(ClTile<2, 1, 2, 1>{});
        case 3: return go(ClTile<1, 2, 2, 1>{});
        case 4: return go(ClTile<2, 1, 4, 1>{});
        default: return go(ClTile<2, 2, 4, 1>{});
    }
}

static bool copy_fits(const nzhip_gemm_desc& d) {
    const int64_t lim = 1 << 29;
    return d.batch_n * d.batch_c == 1 && d.M < (1 << 22) && d.N < (1 << 22) && d.K < (1 << 22) && (d.M + 256) * (d.K + 128) < lim &&
           (d.N + 256) * (d.K + 128) < lim && (d.K + 64) * (d.M + 384) < lim && (d.K + 64) * (d.N + 384) < lim && d.M * d.N < lim && d.ldc < (1 << 22) &&
           d.lda < (1 << 30) && d.ldb < (1 << 30);
}

struct CopyPlan { int tile, parts; };
static bool copy_plan_env(CopyPlan& pl) {
    const char* e = getenv("NZHIP_GEMM_COPY_PLAN");                   // read per call (tests, benchmarking): "tile,parts"
    CopyPlan q;
    if (!e || sscanf(e, "%d,%d", &q.tile, &q.parts) != 2 || q.tile < 0 || q.tile >= COPY_TILES || q.parts < 1) return false;
    pl = q;
    return true;
}

// Estimated time in us and the plan it is for, fitted on 66 products and pairs of 16 to 4096 rows, columns and k with 15 plans each: the plan
// chosen is 1.4 % slower than the best of the 15 in the geometric mean, 13 % at worst. A k step (64) of a workgroup alone on its CU
// takes `alone`, of two that share one `pair` together.
static CopyPlan copy_plan_search(const nzhip_gemm_desc* d, int count, bool one_sum, double* cost) {
    static const double alone[COPY_TILES] = {0.207, 0.482, 0.385, 0.296, 0.530, 0.800}, pair[COPY_TILES] = {0.329, 0.482, 0.453, 0.469, 0.530, 0.800};
    static const double first[COPY_TILES] = {4.4, 4.7, 4.1, 4.3, 5.9, 6.0};      // launch, first request and result of a workgroup
    static const int cuts[] = {1, 2, 3, 4, 6, 8, 12, 16};
    const double cus = device_cu_count();
    double least = 1e30, rounding = 0.0, out = 0.0;
    for (int i = 0; i < count; i++) {
        const double m = (double)d[i].M, n = (double)d[i].N, k = (double)d[i].K;
        rounding += 6.0 * k * (i == 0 ? m + n : n);                  // (the second product's A is the first one's)
        out += m * n * (count == 2 ? 8.0 : 4.0);
    }
    CopyPlan best = {0, 1};
    for (int t = 0; t < COPY_TILES; t++) {
        const CopyShape& sh = COPY_SHAPES[t];
        const bool two = t == 0 || t == 2 || t == 3;
        if (one_sum && sh.kg > 1) continue;
        for (int cut : cuts) {
            if (one_sum && cut > 1) break;
            double wgs = 0.0, work = 0.0, longest = 0.0, summed = 0.0;
            for (int i = 0; i < count; i++) {
                const int64_t steps = (d[i].K + 63) / 64, per = (steps + cut - 1) / cut, parts = (steps + per - 1) / per, own = (per + sh.kg - 1) / sh.kg;
                const double n = (double)((d[i].M + sh.bm - 1) / sh.bm) * (double)((d[i].N + sh.bn - 1) / sh.bn) * (double)parts;
                wgs += n; work += n * (double)own;
                if ((double)own > longest) longest = (double)own;
                if (parts > 1) summed += (double)d[i].M * (double)d[i].N * 4.0 * (2.0 * (double)parts + 1.0);
            }
            if (cut > 1 && (summed == 0.0 || wgs > 8.0 * cus)) break;
            double main = first[t];
            if (wgs <= cus) main += longest * alone[t];
            else {
                const double rounds = wgs / (cus * (two ? 2 : 1)), filled = rounds < 1.0 ? 1.0 : rounds < 3.0 ? std::ceil(rounds) : rounds + 0.4;
                const double share = wgs / cus - 1.0 < 1.0 ? wgs / cus - 1.0 : 1.0, step = two ? alone[t] + (pair[t] - alone[t]) * share : alone[t];
                const double load = filled * work / wgs;
                main += (load > longest ? load : longest) * step + (filled - 1.0) * 2.6;
            }
            main += out / 4.2e6;
            if (summed > 0.0) main += 2.2 + summed / 6.9e6;
            if (main < least) {
                least = main;
                best = {t, cut};
            }
        }
    }
    *cost = 2.8 + rounding / 7.9e6 + least;
    return best;
}

static CopyPlan copy_plan(const nzhip_gemm_desc* d, int count, bool one_sum, double* cost) {
    struct Key { int64_t count, m, n, k, m2, n2, k2; };
    struct Found { CopyPlan plan; double cost; };
    static thread_local PlanCache<Key, Found> cache;
    const bool pair = count == 2;
    const Key key = {count + one_sum * 4 + (int64_t)device_cu_count() * 8, d[0].M, d[0].N, d[0].K, pair ? d[1].M : 0, pair ? d[1].N : 0, pair ? d[1].K : 0};
    bool known;
    Found& f = cache.at(key, known);
    if (!known) f.plan = copy_plan_search(d, count, one_sum, &f.cost);
    if (cost) *cost = f.cost;
    return f.plan;
}

// halfs of the copy of an operand of `rows` rows, a whole number of 128-byte lines
static size_t copy_halfs(int64_t rows, int64_t cols) { return ((size_t)rows * cl_pitch((int)cols) + 63) / 64 * 64; }

// bytes of workspace the products take at most (an operand that both share counted twice)
static size_t copy_bytes(const nzhip_gemm_desc* d, int count, const CopyPlan& pl) {
    size_t bytes = 4096;
    for (int i = 0; i < count; i++) {
        const bool a_kc = d[i].a_layout == NZHIP_LAYOUT_ROW, b_kc = d[i].b_layout == NZHIP_LAYOUT_TRANS;
        bytes += 2 * (a_kc ? copy_halfs(d[i].M, d[i].K) : copy_halfs(d[i].K, d[i].M)) + 2 * (b_kc ? copy_halfs(d[i].N, d[i].K) : copy_halfs(d[i].K, d[i].N));
        if (pl.parts > 1) bytes += (size_t)pl.parts * d[i].M * d[i].N * sizeof(float);
    }
    return bytes;
}

// NZHIP_E_NOMEM: no memory for the copies or partial sums, and nothing was launched
int gemm_copy_run(const nzhip_gemm_desc* d, int count, hipStream_t s, bool one_sum) {
    CopyPlan pl = copy_plan(d, count, one_sum, nullptr);
    copy_plan_env(pl);
    const CopyShape sh = COPY_SHAPES[pl.tile];
    struct Operand { const float* p; int64_t ld, rows, cols; size_t at; int pitch; };
    Operand ops[4];
    int n_ops = 0, which[2][2];
    size_t halfs = 0;
    auto operand = [&](const float* p, int64_t ld, int64_t rows, int64_t cols) {
        for (int i = 0; i < n_ops; i++)
            if (ops[i].p == p && ops[i].ld == ld && ops[i].rows == rows && ops[i].cols == cols) return i;
        ops[n_ops] = {p, ld, rows, cols, halfs, cl_pitch((int)cols)};
        halfs += copy_halfs(rows, cols);
        return n_ops++;
    };
    CopyPair a = {};
    size_t partials = 0;
    int form[2] = {0, 0};
    for (int i = 0; i < count; i++) {
        const nzhip_gemm_desc& g = d[i];
        const bool a_kc = g.a_layout == NZHIP_LAYOUT_ROW, b_kc = g.b_layout == NZHIP_LAYOUT_TRANS;
        form[i] = (a_kc ? 1 : 0) | (b_kc ? 2 : 0);
        which[i][0] = operand(g.A, g.lda, a_kc ? g.M : g.K, a_kc ? g.K : g.M);
        which[i][1] = operand(g.B, g.ldb, b_kc ? g.N : g.K, b_kc ? g.K : g.N);
        CopyProduct& p = a.p[i];
        p.C = g.C; p.bias = g.bias; p.M = (int)g.M; p.N = (int)g.N; p.K = (int)g.K; p.ldc = (int)g.ldc;
        p.bias_sm = g.bias_stride_row; p.bias_sn = g.bias_stride_col; p.relu = g.activation == NZHIP_ACT_RELU;
        const int steps = (p.K + 63) / 64;
        p.part_steps = (steps + pl.parts - 1) / pl.parts;
        p.chain = one_sum ? 1 << 30 : p.M <= 64 || p.N <= 64 ? cl_chain(p.part_steps / sh.kg) : CL_CHAIN;      // narrow ones: the fused kernel's chunks are of 128
        p.parts = (steps + p.part_steps - 1) / p.part_steps;
        p.tiles_m = (p.M + sh.bm - 1) / sh.bm; p.tiles_n = (p.N + sh.bn - 1) / sh.bn;
        p.tiles = p.tiles_m * p.tiles_n;
        p.by_tiles = cl_div(p.tiles); p.by_panel = cl_div(8 * p.tiles_m);
        if (p.parts > 1) partials += (size_t)p.parts * p.M * p.N;
        a.total += p.tiles * p.parts;
    }
    a.longer = count == 2 && a.p[1].part_steps > a.p[0].part_steps;
    a.head = a.p[a.longer].tiles * a.p[a.longer].parts;
    _Float16* copies = nullptr;
    if (int rc = workspace_alloc(reinterpret_cast<void**>(&copies), halfs * 2, s)) return rc;
    float* partial = nullptr;
    int rc = partials ? workspace_alloc(reinterpret_cast<void**>(&partial), partials * sizeof(float), s) : NZHIP_OK;
    auto done = [&](const char* what) {
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? NZHIP_OK : set_hip_error(e, what);
    };
    if (rc == NZHIP_OK) {
        CopyJobs jobs = {};
        int blocks = 0;
        for (int i = 0; i < n_ops; i++) {
            const int units = (int)((ops[i].cols + 7) / 8);
            jobs.job[i] = {ops[i].p, copies + ops[i].at, (long)ops[i].ld, (int)ops[i].rows, (int)ops[i].cols, ops[i].pitch,
                           (int)((ops[i].rows * units + 255) / 256), cl_div(units)};
            blocks += jobs.job[i].blocks;
        }
        hipLaunchKernelGGL(round_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, s, jobs);
        rc = done("round_rows kernel launch");
    }
    if (rc == NZHIP_OK) {
        float* next = partial;
        for (int i = 0; i < count; i++) {
            CopyProduct& p = a.p[i];
            const Operand &oa = ops[which[i][0]], &ob = ops[which[i][1]];
            p.A = copies + oa.at; p.lda = oa.pitch; p.a_bytes = (unsigned)((size_t)oa.rows * oa.pitch * 2);
            p.B = copies + ob.at; p.ldb = ob.pitch; p.b_bytes = (unsigned)((size_t)ob.rows * ob.pitch * 2);
            if (p.parts > 1) {
                p.partial = next;
                next += (size_t)p.parts * p.M * p.N;
            }
        }
        rc = copy_pick(pl.tile, [&](auto tile) {
            using T = decltype(tile);
            auto kfn = count == 2     ? copy_pair_kernel<1, 0, T>
                       : form[0] == 0 ? copy_product_kernel<0, T>
                       : form[0] == 1 ? copy_product_kernel<1, T>
                       : form[0] == 2 ? copy_product_kernel<2, T>
                                      : copy_product_kernel<3, T>;
            if (int lrc = ensure_dynamic_lds(reinterpret_cast<const void*>(kfn), T::RING, "hipFuncSetAttribute(gemm copies)")) return lrc;
            hipLaunchKernelGGL(kfn, dim3((unsigned)a.total), dim3(T::THREADS), T::RING, s, a);
            return done("copy product kernel launch");
        });
    }
    if (rc == NZHIP_OK && partials) {
        const int b1 = a.p[0].parts > 1 ? (a.p[0].M * a.p[0].N + 255) / 256 : 0, b2 = count == 2 && a.p[1].parts > 1 ? (a.p[1].M * a.p[1].N + 255) / 256 : 0;
        hipLaunchKernelGGL(copy_sum_kernel, dim3((unsigned)(b1 + b2)), dim3(256), 0, s, a, b1, cl_div(a.p[0].N), cl_div(count == 2 ? a.p[1].N : 1));
        rc = done("copy sum kernel launch");
    }
    const int rc2 = partial ? workspace_free(partial, s) : NZHIP_OK, rc3 = workspace_free(copies, s);
    return rc ? rc : rc2 ? rc2 : rc3;
}

bool gemm_copy_wanted(const nzhip_gemm_desc* d, int count, double other_us, bool one_sum) {
    const char* env = getenv("NZHIP_GEMM_COPY");                      // read per call (tests, benchmarking): 0 never, 1 wherever it fits
    if (env && !atoi(env)) return false;
    // a run that asks for one of the other routes, or for a plan of theirs, gets it
    static const bool others = getenv("NZHIP_GEMM_ROUTE") || getenv("NZHIP_SPLITK") || getenv("NZHIP_GEMM_TILE") || getenv("NZHIP_GEMM_WAVES");
    if (!env && others) return false;
    for (int i = 0; i < count; i++)
        if (!copy_fits(d[i])) return false;
    if (count == 2 && (d[0].a_layout != NZHIP_LAYOUT_ROW || d[0].b_layout != NZHIP_LAYOUT_ROW || d[1].a_layout != NZHIP_LAYOUT_TRANS ||
                       d[1].b_layout != NZHIP_LAYOUT_ROW)) return false;
    if (!env && count == 1 && d[0].M <= 64 && d[0].N <= 64) return false;      // one tile: the fused kernel is over before a second launch begins (33 x 512 x 33 7.6 us)
    double cost;
    CopyPlan pl = copy_plan(d, count, one_sum, &cost);
    copy_plan_env(pl);
    // The call that allocates nothing has to give the same bits: one product takes this route only where its copies fit that call's
    // scratch as well (one sum over k has the same bits on either route).
    const size_t bytes = copy_bytes(d, count, pl);
    if (bytes > workspace_limit() || (!env && count == 1 && !one_sum && bytes > NZHIP_STATIC_SCRATCH_BYTES)) return false;
    if (env) return true;
    // The other estimate is above the time by a fifth where B is read along its rows, by a twentieth where it is not (69 products of 31 to
    // 6629 rows), and half a us pays for the second launch. Of those 69 the route taken is 1.4 % behind the better one in the geometric
    // mean. Copies ahead: 944 x 2352 x 1984 38.0 -> 25.8 us, 1000 x 777 x 513 14.9 -> 11.5, 261 x 576 x 528 10.8 -> 8.0. Behind, and not taken:
    // 128 x 1024 x 1024 9.3 us or 9.8, 112 x 2721 x 1853 15.3 or 16.7, 1520 x 243 x 346 6.4 or 7.0, 66 x 6196 x 5601 38 or 54.
    if (count == 2) {
        // Two products' operands and results outgrow the caches as they grow, which the steps' times do not know: 12 % at 3e11 flops, 24 % at 2e12.
        // 113 pairs of 256 to 8192 samples, inputs and outputs: one taken is more than 4 % behind two calls, 2560 x 6336 -> 2112 212 / 234. Taken: 4096
        // samples, 1024 inputs, 4096 outputs 168 -> 104 us, 3072^3 205 / 191, 4001^3 420 / 377, 537 x 681 -> 644 28.3 -> 12.4. Not taken: 4096^3
        // 304 / 369, 8192 x 4096 -> 4096 551 / 690, 5000 x 3000 -> 3500 313 / 332, 8192^3 1951 / 2594.
        const double flops = 4.0 * d[0].M * d[0].N * d[0].K;
        return cost * std::max(1.0, 1.0 + 0.045 * std::log2(flops / 5e10)) < other_us;
    }
    return cost + 0.5 < other_us * (d[0].b_layout == NZHIP_LAYOUT_TRANS ? 0.80 : 0.95);
}

}  // namespace nzhip
