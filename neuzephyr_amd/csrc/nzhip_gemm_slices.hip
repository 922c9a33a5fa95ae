// Products of few tiles, in one launch without a workspace: the waves of a workgroup share an output tile and cut the CONTRACTION between them.
//
// Such a product is over in the time of a launch and a handful of requests to memory; what the other kernels spend is a chain of k steps with
// a barrier each (the fused kernel), or a second launch (partial sums, rounded copies). Here every wave takes each 4th or 8th chunk of 32 k
// of one tile, on its own: fp32 from memory to registers, fragments, MFMAs, no barrier and no data of another wave's until the sums meet in LDS
// at the end. A product of 256^3 is 8 chunks, one per wave; half of a wave's cycles there are waits, and the launch is most of the rest. Longer sums are
// bound by what the vector memory path returns to a CU's registers: a k of a 32 x 32 tile, 256 bytes, takes 2.2 to 2.3 ns (the estimate's fit below), 110 GB/s.
// So tiles are 32 x 32 (more CUs) until there are enough of 64 x 64. us a call, calls queued one behind the other, on the kernels before and here:
// 256^3 5.5 / 4.0, 300^3 8.0 / 4.4, 512^3 7.5 / 4.7, 100 x 1000 x 200 10.2 / 5.9, 33 x 512 x 33 9.8 / 4.4, 1024^3 12.7 / 11.5.
#include <hip/hip_runtime.h>

#include <cstdlib>

#include "nzhip_internal.h"
#include "nzhip_lds_tiles.h"
#include "nzhip_pieces.h"
#include "nzhip_slices.h"

namespace nzhip {

struct SliceArgs {
    const float* A;
    const float* B;
    float* C;
    const float* bias;
    int M, N, K, lda, ldb, ldc;
    long a_sn, a_sc, b_sn, b_sc, c_sn, c_sc, bias_sn, bias_sc, bias_sm, bias_sk;
    int relu, tiles_m, tiles_n, tiles, total, batch_c;
    ClDiv by_tiles, by_panel, by_batch_c;
};

// One operand's share of a k32 chunk, in registers as fp32: F blocks of 32 rows (of A, or columns of B). Requests go through a buffer of the
// operand's size, offsets in bytes.
// KC: k runs along its rows in memory; 8 lanes take the 128 bytes of a row, 16 each, and the fragments are formed through LDS.
template <bool KC, int F>
struct Slice {
    static constexpr int PITCH = SLICE_PITCH;
    static constexpr int LDS = F * 32 * PITCH;
    uint4_t v[F * 4];
    unsigned off[F * 4];
    __amdgpu_buffer_rsrc_t from;
    __device__ __forceinline__ void start(const float* x, int ld, int row0, int rows, int K, int lane) {
        from = slice_buffer(x, (unsigned)((rows - 1) * ld + K) * 4u);
#pragma unroll
        for (int p = 0; p < F * 4; p++) {
            const int r = row0 + p * 8 + (lane >> 3);
            off[p] = (unsigned)((r < rows ? r : rows - 1) * ld + (lane & 7) * 4) * 4u;
        }
    }
    // in the last chunk: pieces that the row's end cuts, or that lie past it, start at its last four elements
    static __device__ __forceinline__ int back(int k0, int K, int lane) {
        const int past = k0 + (lane & 7) * 4 + 4 - K;
        return past > 0 ? past : 0;
    }
    __device__ __forceinline__ void load(int k0, int K, int lane) {
        const unsigned add = (unsigned)(k0 - back(k0, K, lane)) * 4u;
#pragma unroll
        for (int p = 0; p < F * 4; p++) v[p] = __builtin_amdgcn_raw_buffer_load_b128(from, off[p] + add, 0, 0);
    }
    __device__ __forceinline__ void convert(half8_t (&)[2][F], char* lds, int k0, int K, int lane, bool) {
        const int at = k0 + (lane & 7) * 4, moved = back(k0, K, lane);
        const bool whole = k0 + 32 <= K;
#pragma unroll
        for (int p = 0; p < F * 4; p++) {
            piece4 q = __builtin_bit_cast(piece4, v[p]);
            if (!whole) {
                q = turn_back(q, moved);
#pragma unroll
                for (int e = 0; e < 4; e++) q[e] = at + e < K ? q[e] : 0.f;
            }
            half4_t h;
#pragma unroll
            for (int e = 0; e < 4; e++) h[e] = (_Float16)q[e];
            *reinterpret_cast<half4_t*>(lds + (p * 8 + (lane >> 3)) * PITCH + (lane & 7) * 8) = h;
        }
    }
    __device__ __forceinline__ void read(half8_t (&h)[2][F], const char* lds, int lane) {
        const char* q = lds + (lane & 31) * PITCH + (lane >> 5) * 16;
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int f = 0; f < F; f++) h[s][f] = *reinterpret_cast<const half8_t*>(q + f * 32 * PITCH + s * 32);
    }
    static __device__ __forceinline__ int row(int f, int i) { return f * 32 + i; }
};
// k runs across its rows: a lane takes its own row's (column's) elements, F neighbours of each of 16 k, which are its fragments. k past the end
// are past the buffer's end, and come back as zeros.
template <int F>
struct Slice<false, F> {
    static constexpr int LDS = 0;
    unsigned v[16][F];
    unsigned off, ld;
    bool moved;
    __amdgpu_buffer_rsrc_t from;
    __device__ __forceinline__ void start(const float* x, int ld_, int row0, int rows, int K, int lane) {
        from = slice_buffer(x, (unsigned)((K - 1) * ld_ + rows) * 4u);
        ld = (unsigned)ld_ * 4u;
        const int r = row0 + (lane & 31) * F, at = F > 1 && r + F > rows ? rows - F : r < rows ? r : rows - 1;       // a pair that the end cuts starts at the last two
        off = (unsigned)at * 4u + (unsigned)(lane >> 5) * 8u * ld;
        moved = r != at;
    }
    __device__ __forceinline__ void load(int k0, int, int) {
        unsigned o = off + (unsigned)k0 * ld;
        asm volatile("" : "+v"(o));                                 // or 16 offsets per operand are kept in registers from chunk to chunk
#pragma unroll
        for (int s = 0; s < 2; s++) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if constexpr (F == 2) {
                    const uint2_t t = __builtin_amdgcn_raw_buffer_load_b64(from, o, 0, 0);
                    v[s * 8 + e][0] = t[0];
                    v[s * 8 + e][F - 1] = t[1];
                } else {
                    v[s * 8 + e][0] = __builtin_amdgcn_raw_buffer_load_b32(from, o, 0, 0);
                }
                o += ld;
            }
            o += 8u * ld;
        }
    }
    __device__ __forceinline__ void convert(half8_t (&h)[2][F], char*, int, int, int, bool inside) {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (F == 2 && !inside && moved) v[s * 8 + e][0] = v[s * 8 + e][F - 1];
#pragma unroll
                for (int f = 0; f < F; f++) h[s][f][e] = (_Float16)__builtin_bit_cast(float, v[s * 8 + e][f]);
            }
    }
    __device__ __forceinline__ void read(half8_t (&)[2][F], const char*, int) {}
    static __device__ __forceinline__ int row(int f, int i) { return i * F + f; }
};

// FM x FN blocks of 32 x 32 per workgroup, NW waves. The sums of a wave's chunks are chains of 64 elements where registers allow (32 x 32 tiles), of
// K / 8 in the 64 x 64 ones, whose K is short: against 64 bits a relative error of 0.8e-7 at K = 1000, 0.7e-7 to 1.5e-7 on the kernels before.
template <int FM, int FN, bool A_KC, bool B_KC, int NW>
__global__ __launch_bounds__(NW * 64, FM * FN == 4 ? 2 : 4) void gemm_slices_kernel(const SliceArgs p) {
    using SA = Slice<A_KC, FM>;
    using SB = Slice<B_KC, FN>;
    constexpr int BM = FM * 32, BN = FN * 32, STAGE = SA::LDS + SB::LDS;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 31, lh = lane >> 5;

    const int lin = cl_xcd_place(blockIdx.x, p.total);
    const int member = cl_quot(lin, p.by_tiles), t = lin - member * p.tiles;
    const int panel = cl_quot(t, p.by_panel), wide = p.tiles_n - panel * 8 < 8 ? p.tiles_n - panel * 8 : 8, in = t - panel * 8 * p.tiles_m;
    const int tile_m = wide == 8 ? in >> 3 : in / wide, tile_n = panel * 8 + in - tile_m * wide;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int bi = cl_quot(member, p.by_batch_c), bj = member - bi * p.batch_c;

    SA sa;
    SB sb;
    sa.start(p.A + bi * p.a_sn + bj * p.a_sc, p.lda, m0, p.M, p.K, lane);
    sb.start(p.B + bi * p.b_sn + bj * p.b_sc, p.ldb, n0, p.N, p.K, lane);
    const bool inside_m = m0 + BM <= p.M, inside_n = n0 + BN <= p.N;
    char* own_a = lds + wave * STAGE;
    char* own_b = own_a + SA::LDS;

    floatx16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    const int chunks = (p.K + 31) >> 5;
    if (wave < chunks) {
        sa.load(wave * 32, p.K, lane);
        sb.load(wave * 32, p.K, lane);
    }
    floatx16 sum[FM][FN];                                           // of the chunks so far but the last two: a chain of 64 elements
    if constexpr (FM * FN == 1) sum[0][0] = acc[0][0];
    int odd = 0;
    for (int c = wave; c < chunks; c += NW) {
        const int k0 = c * 32, k1 = k0 + NW * 32;
        half8_t a[2][FM], b[2][FN];
        sa.convert(a, own_a, k0, p.K, lane, inside_m);
        sb.convert(b, own_b, k0, p.K, lane, inside_n);
        if (c + NW < chunks) {
            sa.load(k1, p.K, lane);
            sb.load(k1, p.K, lane);
        }
        slice_wave_sync();
        sa.read(a, own_a, lane);
        sb.read(b, own_b, lane);
        if (FM * FN == 1 && (odd ^= 1)) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                sum[0][0][r] += acc[0][0][r];
                acc[0][0][r] = 0.f;
            }
        }
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[s][i], b[s][j], acc[i][j], 0, 0, 0);
        slice_wave_sync();
    }

    if constexpr (FM * FN == 1)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[0][0][r] += sum[0][0][r];

    // the waves' sums meet in LDS, four rows of a column at a time
    const int active = chunks < NW ? chunks : NW;
    piece4* park = reinterpret_cast<piece4*>(lds);
    if (STAGE) __syncthreads();
    if (wave < active) slice_park(park, acc, wave, lane);
    __syncthreads();
    float* C = p.C + bi * p.c_sn + bj * p.c_sc;
    const float* bias = p.bias ? p.bias + bi * p.bias_sn + bj * p.bias_sc : nullptr;
#pragma unroll
    for (int q = 0; q < (FM * 4 + NW - 1) / NW; q++) {
        const int ig = wave + q * NW, i = ig >> 2, g = ig & 3;
        if (ig >= FM * 4) break;
        piece4 s[FN];
#pragma unroll
        for (int j = 0; j < FN; j++) s[j] = slice_collect<FM, FN, NW>(park, ig, j, active, lane);
        float bv[4][FN];
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int j = 0; j < FN; j++) {
                const int m = m0 + SA::row(i, g * 8 + lh * 4 + e), n = n0 + SB::row(j, li);
                bv[e][j] = bias ? bias[(m < p.M ? m : 0) * p.bias_sm + (n < p.N ? n : 0) * p.bias_sk] : 0.f;
            }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int m = m0 + SA::row(i, g * 8 + lh * 4 + e);
            if (m >= p.M) continue;
            float o[FN];
#pragma unroll
            for (int j = 0; j < FN; j++) {
                o[j] = s[j][e] + bv[e][j];
                if (p.relu) o[j] = o[j] > 0.f ? o[j] : 0.f;
            }
            const int n = n0 + SB::row(0, li);
            float* to = C + (long)m * p.ldc + n;
            if (FN == 2 && !B_KC && n + 1 < p.N) {
                *reinterpret_cast<floatx2u*>(to) = floatx2u{o[0], o[FN - 1]};
            } else {
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    const int nj = n0 + SB::row(j, li);
                    if (nj < p.N) to[nj - n] = o[j];
                }
            }
        }
    }
}

// ---- host side ----------------------------------------------------------------------------------------------------------
struct SliceShape { int f, nw; };                                    // 32 f x 32 f tiles
constexpr SliceShape SLICES[3] = {{1, 4}, {1, 8}, {2, 8}};

template <int F, int NW>
static int slices_launch(const SliceArgs& a, bool a_kc, bool b_kc, hipStream_t s) {
    auto go = [&](auto kfn, int stage) {
        const int park = NW * F * F * 4096, lds = park > stage * NW ? park : stage * NW;
        if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kfn), lds, "hipFuncSetAttribute(gemm slices)")) return rc;
        hipLaunchKernelGGL(kfn, dim3((unsigned)a.total), dim3(NW * 64), (size_t)lds, s, a);
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? NZHIP_OK : set_hip_error(e, "gemm slices kernel launch");
    };
    constexpr int stage = Slice<true, F>::LDS;
    if (a_kc && b_kc) return go(gemm_slices_kernel<F, F, true, true, NW>, 2 * stage);
    if (a_kc) return go(gemm_slices_kernel<F, F, true, false, NW>, stage);
    if (b_kc) return go(gemm_slices_kernel<F, F, false, true, NW>, stage);
    return go(gemm_slices_kernel<F, F, false, false, NW>, 0);
}

// the extents that the kernel's 32-bit offsets hold; pieces of 4 along k, and pairs across it, want as many
static bool slices_fit(const nzhip_gemm_desc& d, int shape) {
    if (SLICES[shape].f == 2 && (d.M < 2 || d.N < 2)) return false;
    const int64_t lim = 1 << 29, members = d.batch_n * d.batch_c;
    if (d.K < 4 || d.M >= (1 << 22) || d.N >= (1 << 22) || d.K >= (1 << 22) || members > (1 << 20) || d.lda >= lim || d.ldb >= lim || d.ldc >= lim) return false;
    // an operand of up to 2 GiB: its rows, and 64 k past them
    const int64_t ra = d.a_layout == NZHIP_LAYOUT_ROW ? d.M : d.K + 64, rb = d.b_layout == NZHIP_LAYOUT_TRANS ? d.N : d.K + 64;
    return ra * d.lda + d.K < lim && rb * d.ldb + d.K < lim && (d.M / 32 + 1) * (d.N / 32 + 1) * members < (1 << 28);
}

// The shape a product is to run with, -1: another kernel is faster. Drawn on 430 products of 1 to 4096 rows and columns and 16 to 2500 k, and again on 2600
// of 1 to 4 rows or columns and 1900 others, against the kernels that took them before (us there / here):
// - K up to 2048: past that a CU's intake of K x 64 elements outlasts a second launch (80 x 1760 x 288 10.0 / 8.4, 48 x 1943 x 112 9.7 / 7.5; 64 x 1728 x 384
//   9.0 / 8.4, 48 x 2279 x 576 9.4 / 11.9, 11 x 2480 x 1040 8.4 / 9.7).
// - 95 MB that the tiles take in, 130 where both operands run along k, and at most 1024 tiles: 1472 x 231 x 464 8.1 / 6.0, 373 x 704 x 884 10.0 / 7.5,
//   1408 x 640 x 357 11.0 / 9.0, 984 x 1328 x 366 with B along k 12.5 / 11.7; 1000 x 777 x 513 11.5 / 12.4, 601 x 1481 x 485 13.8 / 15.2, 1305 x 409 x 819 (1066 tiles) 10.3 / 11.6.
//   A fourth round of the CUs pays with both operands across k only (3056 x 421 x 304 with both along it, 960 tiles, 8.3 / 9.8, 736 x 639 x 1088 9.7 / 11.4, B along it
//   1135 x 276 x 874 7.5 / 8.1): 768 tiles with both along it, 896 with B alone, 80 MB past 768 with A alone (356 x 426 x 2167, 816 tiles, 9.8 / 11.2).
// - one or two rows or columns whose product only streams the other operand, with a kernel that does no more than that, along k: up to 640 k (378 x 352 x 2 5.8 / 4.9,
//   2 x 528 x 576 5.4 / 4.3; 1 x 1516 x 480 4.5 / 5.9, 18 x 914 x 1 5.9 / 6.4); one row by rows of 16-byte pieces up to 128 (1 x 208 x 2 2.9 / 3.5, 1 x 448 x 263
//   3.6 / 3.9), one column 32 (528 x 256 x 1 3.2 / 4.2, 976 x 368 x 1 3.6 / 4.5; 96 x 16 x 1 3.5 / 3.2), with other rows 384 by up to 64 of them (2 x 465 x 1 3.4 / 4.0;
//   1 x 323 x 128 4.5 / 4.0).
//   Across k the streaming kernel needs a second launch (1 x 832 x 3314 14.9 / 5.9, 288 x 1279 x 2 10.6 / 7.5), but not for a handful of k (195 x 6 x 1 2.8 / 3.4, one row or
//   column of up to 16 in pieces) and not where a workgroup keeps whole columns, up to 4096 of them (2064 x 1136 x 1 4.0 / 6.1, 2 x 1424 x 2688 4.8 / 6.9; 1 x 1760 x 6000 14.7 / 9.0).
// - 64 x 64 tiles where they fill two thirds of the CUs or more, in one round: 1378 x 690 x 448 10.9 / 8.6, 1344 x 864 x 624 11.7 / 10.8, 541 x 1472 x 1232
//   15.9 / 14.2, 1024^3 13.5 / 11.7; 572 x 1024 x 1153 12.2 / 12.2, 727 x 1289 x 752 (144 tiles) 13.3 / 15.7, 1221 x 816 x 848 (280) 14.4 / 20.9. With both operands along k
//   up to 1280 k (588 x 1441 x 1136 14.9 / 16.9, 991 x 1507 x 650 15.9 / 17.0), and not whole tiles, on which the fused kernel is at its best (1024^3 10.2 / 11.6).
static int slices_shape(const nzhip_gemm_desc& d) {
    const int64_t members = d.batch_n * d.batch_c, lo = d.M < d.N ? d.M : d.N;
    const bool a_kc = d.a_layout == NZHIP_LAYOUT_ROW, b_kc = d.b_layout == NZHIP_LAYOUT_TRANS;
    const int64_t t32 = (d.M + 31) / 32 * ((d.N + 31) / 32) * members, t64 = (d.M + 63) / 64 * ((d.N + 63) / 64) * members;
    const int cus = device_cu_count();
    if (d.K > 2048) return -1;
    if (lo <= 2) {
        const int64_t hi = d.M < d.N ? d.N : d.M;
        const SkinnyForm f = gemm_skinny_form(d);
        if (d.K > 640 && (f.along || hi == 1)) return -1;
        if (f.along && lo == 1 && (f.pieces ? d.K > (d.N == 1 ? 32 : 128) : d.K > 384 && hi <= 64)) return -1;
        if (!f.along && (d.K < 10 || (lo == 1 && f.pieces && d.K <= 16) || (f.columns && hi <= 4096))) return -1;
    }
    const int64_t most = !b_kc ? 1024 : a_kc ? 768 : 896, in = a_kc && b_kc ? 130000000 : a_kc && t32 > 768 ? 80000000 : 95000000;
    // more tiles than CUs: workgroups of 4 waves, of which a CU holds more (1500 x 250 x 350 6.3 us with 4, 8.2 with 8)
    if (t32 <= most && t32 * d.K * 256 <= in) return t32 > cus || d.K <= 128 ? 0 : 1;
    if (lo > 2 && t64 <= cus && t64 * 3 >= cus * 2 && d.K <= (a_kc && b_kc ? 1280 : 1536) && !(a_kc && b_kc && (d.M | d.N | d.K) % 64 == 0)) return 2;
    return -1;
}

int gemm_slices_plan(const nzhip_gemm_desc& d) {
    static const bool others = getenv("NZHIP_GEMM_ROUTE") || getenv("NZHIP_SPLITK") || getenv("NZHIP_GEMM_TILE") || getenv("NZHIP_GEMM_WAVES") || getenv("NZHIP_SKINNY_MAX");
    const char* env = getenv("NZHIP_GEMM_SLICES");                    // read per call (tests, benchmarking): 0 never, 1 to 3 that shape wherever it fits
    if (env) {
        const int shape = atoi(env) - 1;
        return shape >= 0 && shape < 3 && slices_fit(d, shape) ? shape : -1;
    }
    if (others || getenv("NZHIP_GEMM_COPY")) return -1;               // a run that asks for one of the other routes gets it
    const int shape = slices_shape(d);
    return shape >= 0 && slices_fit(d, shape) ? shape : -1;
}

// Estimated time in us of a product that is added to what is there, fitted on 1260 of a Linear layer's gradients (700 layers of 4 to 2048 samples, 5 % off on average)
double gemm_slices_cost(const nzhip_gemm_desc& d, int shape) {
    const bool a_kc = d.a_layout == NZHIP_LAYOUT_ROW;
    const int side = 32 * SLICES[shape].f;
    const double tiles = (double)((d.M + side - 1) / side) * (double)((d.N + side - 1) / side) * (double)(d.batch_n * d.batch_c) / device_cu_count();
    const double k = (double)d.K * (tiles > 1.0 ? tiles : 1.0), out = (double)d.M * (double)d.N * (double)(d.batch_n * d.batch_c) * 1e-6;
    if (shape == 0) return a_kc ? 3.47 + 0.0040 * k + 1.2 * out : 3.25 + 0.0034 * k + 1.2 * out;
    if (shape == 1) return a_kc ? 3.69 + 0.0023 * (double)d.K + 2.1 * out : 3.24 + 0.0022 * (double)d.K + 2.9 * out;
    return 5.4 + 0.0058 * k + 2.0 * out + (tiles > 1.0 ? 9.7 * (tiles - 1.0) : 0.0);
}

int gemm_slices_run(const nzhip_gemm_desc& d, int shape, hipStream_t s) {
    const SliceShape sh = SLICES[shape];
    SliceArgs a = {};
    a.A = d.A; a.B = d.B; a.C = d.C; a.bias = d.bias;
    a.M = (int)d.M; a.N = (int)d.N; a.K = (int)d.K; a.lda = (int)d.lda; a.ldb = (int)d.ldb; a.ldc = (int)d.ldc;
    a.a_sn = d.a_stride_n; a.a_sc = d.a_stride_c; a.b_sn = d.b_stride_n; a.b_sc = d.b_stride_c; a.c_sn = d.c_stride_n; a.c_sc = d.c_stride_c;
    a.bias_sn = d.bias_stride_n; a.bias_sc = d.bias_stride_c; a.bias_sm = d.bias_stride_row; a.bias_sk = d.bias_stride_col;
    a.relu = d.activation == NZHIP_ACT_RELU;
    a.tiles_m = (a.M + sh.f * 32 - 1) / (sh.f * 32); a.tiles_n = (a.N + sh.f * 32 - 1) / (sh.f * 32);
    a.tiles = a.tiles_m * a.tiles_n; a.batch_c = (int)d.batch_c; a.total = a.tiles * (int)(d.batch_n * d.batch_c);
    a.by_tiles = cl_div(a.tiles); a.by_panel = cl_div(8 * a.tiles_m); a.by_batch_c = cl_div(a.batch_c);
    const bool a_kc = d.a_layout == NZHIP_LAYOUT_ROW, b_kc = d.b_layout == NZHIP_LAYOUT_TRANS;
    switch (shape) {
        case 0: return slices_launch<1, 4>(a, a_kc, b_kc, s);
        case 1: return slices_launch<1, 8>(a, a_kc, b_kc, s);
        default: return slices_launch<2, 8>(a, a_kc, b_kc, s);
    }
}

}  // namespace nzhip
