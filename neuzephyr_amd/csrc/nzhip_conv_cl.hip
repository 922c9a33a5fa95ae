// Convolutions on channel-last fp16 copies of their operands.
//
// The other Conv2d kernels round the fp32 planes where they stage them, image by image and window by window; on layers that leave
// them few windows (14 x 14 images, 7 x 7 kernels, stride 2) that staging is a serial chain. Here ONE small launch
// (cl_prep_kernel) rounds everything first: x to [image][row][column][channels], surrounded by the zeros of the padding,
// the weights to [output channel][tap][channels], channels padded with zeros to a multiple of 8. What is left is a plain
// matrix product whose operand rows are gathered:
//     y[o][pixel] = sum over (tap, channel) of w[o][tap][channel] * x[base(pixel) + offset(tap)][channel]
// A unit is 8 channels of one tap, 16 bytes in either operand; a k step is 8 units. Tiles go from memory to LDS without
// registers (buffer_load ... lds, 16 bytes a lane, a ring of stages), with no bounds in the loop: padding is in the copy,
// rows past the end repeat the last one. The data gradient is the same sum over the output gradient, one per remainder of
// (row, column) modulo the stride, each with the taps that reach it, so a strided layer multiplies no zeros. The weight gradient
// contracts over the pixels, which are the LDS rows there: its fragments are read through the transposing LDS load.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <type_traits>

#include "nzhip_conv_cl.h"
#include "nzhip_internal.h"
#include "nzhip_lds_tiles.h"
#include "nzhip_pieces.h"
#include "nzhip_plan_cache.h"

namespace nzhip {

// ---- the copies ------------------------------------------------------------------------------------------------
// One job turns `images` sets of (channel, pixel) planes into channel-last rows: pixel p of image i, channel c is read at
//   src + (i / T) * s1 + (i % T) * s2 + c * sc + (p's place in an H x W plane)
// and written, with channels C..Cp-1 zero, to dst + (i / T) * d1 + (i % T) * d2 + p * dp + c. p runs over Hp x Wp pixels of which
// H x W from (pt, pl) on are read and the others are zero. Jobs with `rows` copy rows of C contiguous elements to rows of Cp.
struct ClPrepJob {
    const float* src;
    _Float16* dst;
    long s1, s2, sc, d1, d2, dp;
    int T, C, Cp, H, W, Hp, Wp, pt, pl;
    int ptiles, ctiles, blocks, rows;
};
struct ClPrepArgs { ClPrepJob job[2]; };
constexpr int CLP_PX = 64, CLP_CH = 64, CLP_PITCH = CLP_CH * 2 + 16;

// Bound by memory and, on the small layers it is for, by its launch (4 us). 64 pixels x 64 channels per workgroup: reads run along the
// pixels (256 bytes a wave), the tile is turned in LDS, writes run along the channels (128 bytes a pixel).
__global__ __launch_bounds__(256) void cl_prep_kernel(const ClPrepArgs a) {
    __shared__ __attribute__((aligned(16))) char tile[CLP_PX * CLP_PITCH];
    int b = blockIdx.x;
    const bool second = b >= a.job[0].blocks;
    if (second) b -= a.job[0].blocks;
    const ClPrepJob& j = a.job[second];
    const int tid = threadIdx.x;
    if (j.rows) {                                                 // rows of contiguous elements: only rounded
        const int upr = j.Cp / 8;
        const long u = (long)b * 256 + tid, row = u / upr;
        const int c = (int)(u - row * upr) * 8;
        if (row >= (long)j.rows) return;
        const float* s = j.src + row * j.C + c;
        half8_t h;
        if (c + 8 <= j.C) {
            const piece4 lo = *reinterpret_cast<const floatx4u*>(s), hi = *reinterpret_cast<const floatx4u*>(s + 4);
#pragma unroll
            for (int e = 0; e < 4; e++) { h[e] = (_Float16)lo[e]; h[4 + e] = (_Float16)hi[e]; }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) h[e] = c + e < j.C ? (_Float16)s[e] : (_Float16)0.f;
        }
        const long set = row / j.T;
        *reinterpret_cast<half8_t*>(j.dst + set * j.dp + (row - set * j.T) * j.Cp + c) = h;
        return;
    }
    const int per = j.ptiles * j.ctiles;
    const int img = b / per, rest = b - img * per, ct = rest / j.ptiles, pt = rest - ct * j.ptiles;
    const int c0 = ct * CLP_CH, cn = (j.Cp - c0 < CLP_CH ? j.Cp - c0 : CLP_CH) / 8;       // groups of 8 channels
    const float* src = j.src + (img / j.T) * j.s1 + (img % j.T) * j.s2;
    _Float16* dst = j.dst + (img / j.T) * j.d1 + (img % j.T) * j.d2;
    const int pixels = j.Hp * j.Wp;
    {
        const int px = tid & 63, p = pt * CLP_PX + px;
        const int hp = p / j.Wp, h = hp - j.pt, w = p - hp * j.Wp - j.pl;
        const bool in = p < pixels && (unsigned)h < (unsigned)j.H && (unsigned)w < (unsigned)j.W;
        const float* s = src + (in ? (long)h * j.W + w : 0);
        float v[2][8];
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int c = c0 + ((tid >> 6) + q * 4) * 8 + e;
                v[q][e] = s[(c < j.C ? c : 0) * j.sc];
            }
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int g = (tid >> 6) + q * 4;
            half8_t h8;
#pragma unroll
            for (int e = 0; e < 8; e++) h8[e] = in && c0 + g * 8 + e < j.C ? (_Float16)v[q][e] : (_Float16)0.f;
            if (g < cn) *reinterpret_cast<half8_t*>(tile + px * CLP_PITCH + g * 16) = h8;
        }
    }
    __syncthreads();
    for (int u = tid; u < CLP_PX * cn; u += 256) {
        const int px = u / cn, g = u - px * cn, p = pt * CLP_PX + px;
        if (p < pixels) *reinterpret_cast<half8_t*>(dst + (long)p * j.dp + c0 + g * 8) = *reinterpret_cast<const half8_t*>(tile + px * CLP_PITCH + g * 16);
    }
}

static void prep_planes(ClPrepJob& j, const float* src, _Float16* dst, long images, int C, int Cp, int H, int W, int Hp, int Wp, int pt, int pl) {
    j = {};
    j.src = src; j.dst = dst;
    j.T = 1; j.C = C; j.Cp = Cp; j.H = H; j.W = W; j.Hp = Hp; j.Wp = Wp; j.pt = pt; j.pl = pl;
    j.s1 = (long)C * H * W; j.sc = (long)H * W;
    j.dp = cl_pitch(C); j.d1 = (long)Hp * Wp * j.dp;
    j.ptiles = (Hp * Wp + CLP_PX - 1) / CLP_PX; j.ctiles = (Cp + CLP_CH - 1) / CLP_CH;
    j.blocks = (int)(images * j.ptiles * j.ctiles);
}
// weights [copy][(c, tap)][o] -> [copy][o][tap][Cp]
static void prep_weights(ClPrepJob& j, const float* src, _Float16* dst, long copies, int C, int Cp, int taps, int O) {
    j = {};
    j.src = src; j.dst = dst;
    j.T = taps; j.C = C; j.Cp = Cp; j.H = 1; j.W = O; j.Hp = 1; j.Wp = O;
    j.s1 = (long)C * taps * O; j.s2 = O; j.sc = (long)taps * O;
    j.dp = cl_pitch(taps * Cp); j.d1 = (long)O * j.dp; j.d2 = Cp;
    j.ptiles = (O + CLP_PX - 1) / CLP_PX; j.ctiles = (Cp + CLP_CH - 1) / CLP_CH;
    j.blocks = (int)(copies * taps * j.ptiles * j.ctiles);
}
// sets of `taps` rows of C elements -> the set's rows of Cp one after the other
static void prep_rows(ClPrepJob& j, const float* src, _Float16* dst, long rows, int taps, int C, int Cp) {
    j = {};
    j.src = src; j.dst = dst;
    j.T = taps; j.C = C; j.Cp = Cp; j.rows = (int)rows; j.dp = cl_pitch(taps * Cp);
    j.blocks = (int)((rows * (Cp / 8) + 255) / 256);
}
static int prep_launch(const ClPrepArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(cl_prep_kernel, dim3((unsigned)(a.job[0].blocks + a.job[1].blocks)), dim3(256), 0, s, a);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? NZHIP_OK : set_hip_error(e, "cl_prep kernel launch");
}

// ---- forward and data gradient --------------------------------------------------------------------------------------
constexpr int CL_MAX_CLASSES = 9;                                   // stride^2 sums of a data gradient, 1 of a forward

struct ClClass {
    int nr, ns, r0, rs, s0, ss;         // taps (r0 + i rs, s0 + j ss), i < nr, j < ns
    int di, dj;                         // copy offset of tap (i, j): i di + j dj elements
    int Hc, Wc, base;                   // pixels per image, copy offset of pixel (0, 0) in elements
    int out, out_h, out_w;              // place of pixel (i, j) in its output plane: out + i out_h + j out_w
    int lo_h, lo_w;                     // tap (i, j) of pixel (k, l) reads row lo_h + k - i, column lo_w + l - j of dy (a data gradient)
    ClDiv by_ns, by_hw, by_w;           // ns, Hc Wc, Wc
};
struct ClArgs {
    const _Float16* w;
    const _Float16* x;
    float* y;
    const float* bias;
    float* partial;                     // [part][output] bare sums, or null
    int M, w_row, cu, Kw;               // output channels; weight row in elements; units per tap; taps per tap row
    int step_h, step_w;                 // copy offset between pixel rows / columns of a class, elements
    unsigned w_bytes, x_bytes;          // of one weight copy; of the images one launch row covers
    long x_img, w_img, y_img;           // elements per image
    int images;                         // images in one launch row: N, or 1 with a weight copy per image
    long plane, y_total;                // output plane; elements of y
    long bias_sp, bias_sc, bias_sn;
    int relu, parts, part_units, tiles_m, tiles, n_classes;      // tiles: of all classes or pairs, as if each had as many as the largest
    int paired;                         // classes 2 i and 2 i + 1 are the even and the odd columns of the same rows, and one workgroup's
    int dy_h, dy_w;                     // dy's extents; 0 in a forward
    int units;                          // of the longest sum (host)
    int early_bias;                     // requested before the first step
    ClDiv by_cu, by_tiles_m, by_groups;     // groups: the classes, or the pairs of them
    ClClass cls[CL_MAX_CLASSES];
};

// Units u_first .. + n_units of one element of a data gradient, taps outside dy left out: the zeros around dy are no terms of the sum, and
// times an infinite weight they are not nothing either.
__device__ __forceinline__ float cl_terms(const ClArgs& p, const ClClass& c, const int z, const int img, const int i, const int j, const int o,
                                          const int u_first, const int n_units) {
    const _Float16* x = p.x + z * p.x_img + img * p.x_img + c.base + (long)i * p.step_h + (long)j * p.step_w;
    const _Float16* w = p.w + z * p.w_img + (long)o * p.w_row;
    float s = 0.f;
#pragma unroll 1
    for (int u = u_first; u < u_first + n_units; u++) {
        const int t = cl_quot(u, p.by_cu), ti = cl_quot(t, c.by_ns), tj = t - ti * c.ns, e = (u - t * p.cu) * 8;
        if ((unsigned)(c.lo_h + i - ti) >= (unsigned)p.dy_h || (unsigned)(c.lo_w + j - tj) >= (unsigned)p.dy_w) continue;
        const half8_t a = *reinterpret_cast<const half8_t*>(w + ((c.r0 + ti * c.rs) * p.Kw + c.s0 + tj * c.ss) * p.cu * 8 + e);
        const half8_t b = *reinterpret_cast<const half8_t*>(x + (long)ti * c.di + (long)tj * c.dj + e);
#pragma unroll
        for (int q = 0; q < 8; q++) s = __builtin_fmaf((float)a[q], (float)b[q], s);
    }
    return s;
}

// 64 TM output channels x 32 WN TN pixels per workgroup, 2 x WN waves of 32 TM x 32 TN per k group; KG groups take alternate
// k steps into rings of their own and meet in LDS at the end, where a layer gives fewer tiles than CUs.
// LDS rows are 128 bytes, 8 units; unit u of row r lies at u ^ (r >> 1 & 7), which puts the 16 rows that share a pass of a
// 128-bit read on 16 bank groups. The lane that loads a slot asks for the unit that belongs there, so a lane needs the
// offsets of two units per step (rows of even and odd groups of 8), from a table in LDS, one step ahead.
// DATA: a data gradient. MANY: more than one class. PAIRED: a workgroup has the even columns of its rows and then the odd ones: one run of k steps, two
// sums, stores of two neighbours.
template <typename T, bool DATA, bool MANY, bool PAIRED>
__global__ __launch_bounds__(T::THREADS, 2) void cl_conv_kernel(const ClArgs p) {
    constexpr int TM = T::TM, TN = T::TN, KG = T::KG, BM = T::BM, BN = T::BN, NST = T::NST, STAGE = T::STAGE, LA = T::LA, LB = T::LB, LOADS = LA + LB;
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & (2 * T::WN - 1), kg = KG > 1 ? __builtin_amdgcn_readfirstlane(tid / T::GROUP) : 0;
    const int wm = wave / T::WN, wn = wave % T::WN, li = lane & 31, lh = lane >> 5;

    const int lin = cl_xcd_place(blockIdx.x, p.tiles);
    int ci = 0, in_class = lin;
    // The classes of a strided data gradient take turns: each writes every stride-th pixel of dx, so that the workgroups which write the
    // same lines run together and the L2 of their XCD writes whole ones (16 x 64 x 128 x 128 <- 128 61.6 -> 42.8 us, 16 x 128 x 56 x 56 <- 128
    // 31.4 -> 23.5, against one class after the other). Every second run of eight is reversed: a CU gets each 32nd workgroup of
    // its XCD, and would get only long sums or only short ones (45.3 -> 42.8, 21.0 -> 19.3 on 16 x 256 x 28 x 28 <- 256).
    if (MANY) {
        const int groups = PAIRED ? p.n_classes / 2 : p.n_classes;
        in_class = cl_quot(lin, p.by_groups);
        ci = lin - in_class * groups;
        if (in_class & 8) ci = groups - 1 - ci;
        if (PAIRED) ci *= 2;
    }
    const ClClass& c = p.cls[MANY ? ci : 0];
    const ClClass& odd = p.cls[PAIRED ? ci + 1 : 0];                // as many rows, as many columns or one less: that one's sums are not stored
    const int tile_n = cl_quot(in_class, p.by_tiles_m), tile_m = in_class - tile_n * p.tiles_m;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int z = blockIdx.z;
    const int hw = c.Hc * c.Wc, pixels = p.images * hw;
    if (MANY && n0 >= pixels) return;                               // a class of fewer tiles than the largest

    // units of this part, a whole number of steps per group; the table of their offsets in the two copies, in bytes
    const int u_first = blockIdx.y * p.part_units;
    auto part_of = [&](const ClClass& d) {                          // 0 or less: an empty sum
        const int units = d.nr * d.ns * p.cu;
        return u_first + p.part_units < units ? p.part_units : units - u_first;
    };
    const int n_units = part_of(c), n_odd = PAIRED ? part_of(odd) : 0;
    const int steps = n_units > 0 ? ((n_units + 7) / 8 + KG - 1) / KG : 0, steps_odd = n_odd > 0 ? ((n_odd + 7) / 8 + KG - 1) / KG : 0;
    int2* tab = reinterpret_cast<int2*>(lds + KG * NST * STAGE);
    auto unit_at = [&](int v, const ClClass& d, int n, int shift) {
        const int u = u_first + v, t = cl_quot(u, p.by_cu), i = cl_quot(t, d.by_ns), j = t - i * d.ns, e = (u - t * p.cu) * 8;
        const bool in = v < n;
        return int2{in ? (((d.r0 + i * d.rs) * p.Kw + d.s0 + j * d.ss) * p.cu * 8 + e) * 2 : (int)CL_OUT,
                    in ? (i * d.di + j * d.dj + e + shift) * 2 : (int)CL_OUT};
    };
    for (int v = tid; v < (steps + steps_odd + NST) * KG * 8; v += T::THREADS) {
        const int past = v - steps * KG * 8;
        tab[v] = PAIRED && past >= 0 ? unit_at(past, odd, n_odd, odd.base - c.base) : unit_at(v, c, n_units, 0);
    }

    const int4_t rw = cl_buffer(p.w + z * p.w_img, p.w_bytes), rx = cl_buffer(p.x + z * p.x_img, p.x_bytes);
    unsigned row_a[LA], row_b[LB];
#pragma unroll
    for (int j = 0; j < LA; j++) {
        const int r = m0 + (wave * LA + j) * 8 + (lane >> 3);
        row_a[j] = (unsigned)(r < p.M ? r : p.M - 1) * (unsigned)p.w_row * 2u;
    }
#pragma unroll
    for (int j = 0; j < LB; j++) {
        int px = n0 + (wave * LB + j) * 8 + (lane >> 3);
        if (px >= pixels) px = pixels - 1;
        const int img = cl_quot(px, c.by_hw), q = px - img * hw, i = cl_quot(q, c.by_w), k = q - i * c.Wc;
        row_b[j] = (unsigned)(img * (int)p.x_img + c.base + i * p.step_h + k * p.step_w) * 2u;
    }

    // the results: lane = pixel, registers = channels (r >> 2) * 8 + lh * 4 + (r & 3)
    unsigned out[TN];
    long bpix[TN];
    bool live[TN], both[TN];                                        // both: the odd column's neighbour too
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int px = n0 + (wn * TN + j) * 32 + li;
        live[j] = px < pixels;
        const int pc = live[j] ? px : pixels - 1, img = cl_quot(pc, c.by_hw), q = pc - img * hw, i = cl_quot(q, c.by_w), k = q - i * c.Wc;
        const int pl = c.out + i * c.out_h + k * c.out_w;
        both[j] = PAIRED && live[j] && k < odd.Wc;
        out[j] = (unsigned)((z + img) * (int)p.y_img + pl);
        bpix[j] = (long)(z + img) * p.bias_sn + pl * p.bias_sp;
    }
    const bool split = p.parts > 1;
    float* y = split ? p.partial + blockIdx.y * p.y_total : p.y;
    // The bias of a forward of up to two workgroups a CU is requested before the first step: after the last one it was a trip to memory between
    // the sums and their stores (16 x 256 x 14 x 14 -> 256 18.0 -> 17.4 us a call, 4 x 87 x 59 x 59 -> 50 14.3 -> 13.5; 36 layers 1.5 % in the geometric
    // mean). With more, others cover that trip and first steps would wait for it (16 x 16 x 48 x 48 -> 135 21.3, asked for by all waves at the start
    // 23.8), and waves without a result must not ask (32 x 48 x 51 x 51 -> 16 7x7 25.8 -> 27). The old values of a weight gradient, twice the registers,
    // gained nothing that way (0 to 4 %, but 16 x 100 x 20 x 20 -> 200 with a copy per image 21.0 -> 22.2).
    float bias[DATA ? 1 : TM][DATA ? 1 : TN][16];
    auto request_bias = [&] {
        if constexpr (!DATA) {
            const bool quads = p.bias_sc == 1;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const int o = m0 + (wm * TM + i) * 32 + g * 8 + lh * 4;
                        if (quads && o + 4 <= p.M) {
                            const piece4 v = *reinterpret_cast<const floatx4u*>(p.bias + bpix[j] + o);
#pragma unroll
                            for (int e = 0; e < 4; e++) bias[i][j][g * 4 + e] = v[e];
                        } else {
#pragma unroll
                            for (int e = 0; e < 4; e++) bias[i][j][g * 4 + e] = p.bias[bpix[j] + (long)(o + e < p.M ? o + e : p.M - 1) * p.bias_sc];
                        }
                    }
        }
    };
    if (p.early_bias && kg == 0 && m0 + wm * TM * 32 < p.M) request_bias();

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    char* ring = lds + kg * NST * STAGE;
    const unsigned ring_at = cl_lds(ring) + wave * LA * 1024;
    const int2* slot_unit = tab + kg * 8 + ((lane & 7) ^ (lane >> 4));   // unit of this lane's slot in even groups of 8 rows
    const int2* slot_unit_odd = tab + kg * 8 + ((lane & 7) ^ (lane >> 4) ^ 4);
    int2 next[2];
    auto look_up = [&](int step) {
        next[0] = slot_unit[step * KG * 8];
        next[1] = slot_unit_odd[step * KG * 8];
    };
    auto request = [&](int slot) {
        const unsigned sa = ring_at + slot * STAGE, sb = ring_at + slot * STAGE + BM * 128 + wave * (LB - LA) * 1024;
#pragma unroll
        for (int j = 0; j < LA; j++) cl_load(rw, sa + j * 1024, row_a[j] + next[j & 1].x);
#pragma unroll
        for (int j = 0; j < LB; j++) cl_load(rx, sb + j * 1024, row_b[j] + next[j & 1].y);
    };
    const int sw = (li >> 1) & 7;
    // One step: every fragment is requested before the first MFMA (a read takes 100 clocks and more to come back, an MFMA 32), then
    // the offsets of the next request.
    ClSums<TM, TN> sums;
    auto multiply = [&](const char* base, int t, int chain, int ahead) {
        half8_t af[4][TM], bf[4][TN];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int off = (((k << 1) | lh) ^ sw) << 4;
#pragma unroll
            for (int i = 0; i < TM; i++) af[k][i] = *reinterpret_cast<const half8_t*>(base + ((wm * TM + i) * 32 + li) * 128 + off);
#pragma unroll
            for (int j = 0; j < TN; j++) bf[k][j] = *reinterpret_cast<const half8_t*>(base + BM * 128 + ((wn * TN + j) * 32 + li) * 128 + off);
            __builtin_amdgcn_sched_barrier(0);                      // in the order of their use
        }
        look_up(ahead);
        sums.take(acc, t, chain);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[k][i], bf[k][j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };

    floatx16 even[PAIRED ? TM : 1][PAIRED ? TN : 1];                 // sums of the even columns
    if (steps + steps_odd > 0) {
        __syncthreads();                                            // the table
        // Units past the end are offsets outside both buffers: zeros, in the last step and in requests nobody reads, so the
        // number in flight is the same in every step and no step is special.
        for (int t = 0; t < NST - 1; t++) {
            look_up(t);
            request(t);
        }
        look_up(NST - 1);
        int slot = 0;
        auto run = [&](int from, int n) {
            const int chain = cl_chain(n);
            for (int t = 0; t < n; t++) {
                cl_wait_vmcnt<(NST - 2) * LOADS>();                 // this wave's share of the step has landed
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // everybody's has, and the step before is read by all
                request(slot == 0 ? NST - 1 : slot - 1);
                multiply(ring + slot * STAGE, t, chain, from + t + NST);
                slot = slot == NST - 1 ? 0 : slot + 1;
            }
            sums.finish(acc);
        };
        run(0, steps);
        if constexpr (PAIRED) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        even[i][j][r] = acc[i][j][r];
                        acc[i][j][r] = sums.sum[i][j][r] = 0.f;
                    }
            run(steps, steps_odd);
        }
        cl_wait_vmcnt<0>();
    } else if constexpr (PAIRED) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) even[i][j][r] = 0.f;
    }

    if constexpr (KG > 1) {
        static_assert(KG == 2, "two groups meet pairwise");
        __syncthreads();
        floatx16* park = reinterpret_cast<floatx16*>(lds) + (wave * TM * TN * (PAIRED ? 2 : 1)) * 64 + lane;
        if (kg == 1) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    park[(i * TN + j) * 64] = acc[i][j];
                    if constexpr (PAIRED) park[(TM * TN + i * TN + j) * 64] = even[i][j];
                }
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
                if constexpr (PAIRED) {
                    const floatx16 e = park[(TM * TN + i * TN + j) * 64];
#pragma unroll
                    for (int r = 0; r < 16; r++) even[i][j][r] += e[r];
                }
            }
    }

    if (m0 + wm * TM * 32 >= p.M) return;                           // nothing of this wave's is stored

    // ---- epilogue
    // AGAIN: NaNs of pixels with taps outside dy may come from an infinite weight times the zeros there, and are summed again.
    // d: the class whose sums acc are, `by` columns right of the pixel at out[j]
    auto finish = [&](auto again_tag, const ClClass& d, floatx16 (&acc)[TM][TN], const bool (&live)[TN], const int by, const int n_units) {
        constexpr bool AGAIN = decltype(again_tag)::value;
        unsigned again[TM][TN];
        if (AGAIN)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int px = n0 + (wn * TN + j) * 32 + li, q = px - cl_quot(px, c.by_hw) * hw, h = cl_quot(q, c.by_w), row = d.lo_h + h, col = d.lo_w + q - h * c.Wc;
                const bool edge = live[j] && (row >= p.dy_h || row < d.nr - 1 || col >= p.dy_w || col < d.ns - 1);
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    again[i][j] = 0;
#pragma unroll
                    for (int r = 0; r < 16; r++) again[i][j] |= edge && acc[i][j][r] != acc[i][j][r] ? 1u << r : 0u;
                }
            }
        if (p.bias && !split) {
            if (!p.early_bias) request_bias();
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        if constexpr (DATA) {
                            const int o = m0 + (wm * TM + i) * 32 + (r >> 2) * 8 + lh * 4 + (r & 3);
                            acc[i][j][r] += p.bias[bpix[j] + (live[j] ? by : 0) + (long)(o < p.M ? o : p.M - 1) * p.bias_sc];
                        } else acc[i][j][r] += bias[i][j][r];
                    }
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int o = m0 + (wm * TM + i) * 32 + (r >> 2) * 8 + lh * 4 + (r & 3);
                    float v = acc[i][j][r];
                    if (p.relu && !split) v = v > 0.f ? v : 0.f;
                    if (live[j] && o < p.M && !(AGAIN && again[i][j] >> r & 1)) y[out[j] + by + (unsigned)o * (unsigned)p.plane] = v;
                }
        if (AGAIN)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll 1
                    for (unsigned left = again[i][j]; left; left &= left - 1) {
                        const int r = __builtin_ctz(left), o = m0 + (wm * TM + i) * 32 + (r >> 2) * 8 + lh * 4 + (r & 3);
                        if (o >= p.M) continue;
                        const int px = n0 + (wn * TN + j) * 32 + li, img = cl_quot(px, c.by_hw), q = px - img * hw, h = cl_quot(q, c.by_w);
                        float v = cl_terms(p, d, z, img, h, q - h * c.Wc, o, u_first, n_units);
                        if (p.bias && !split) v += p.bias[bpix[j] + by + o * p.bias_sc];
                        y[out[j] + by + (unsigned)o * (unsigned)p.plane] = v;
                    }
    };
    if constexpr (DATA) {
        float all = 0.f;                                            // NaN if one of them is
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) all += PAIRED ? acc[i][j][r] + even[i][j][r] : acc[i][j][r];
        if (__builtin_expect(__any(all != all), 0)) {
            if constexpr (PAIRED) {
                finish(std::true_type{}, c, even, live, 0, n_units);
                return finish(std::true_type{}, odd, acc, both, 1, n_odd);
            } else return finish(std::true_type{}, c, acc, live, 0, n_units);
        }
    }
    if constexpr (PAIRED) {
        if (p.bias && !split) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int o = m0 + (wm * TM + i) * 32 + (r >> 2) * 8 + lh * 4 + (r & 3);
                        const float* b = p.bias + bpix[j] + (long)(o < p.M ? o : p.M - 1) * p.bias_sc;
                        even[i][j][r] += b[0];
                        acc[i][j][r] += b[both[j] ? 1 : 0];
                    }
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int o = m0 + (wm * TM + i) * 32 + (r >> 2) * 8 + lh * 4 + (r & 3);
                    float* to = y + out[j] + (unsigned)o * (unsigned)p.plane;
                    if (o >= p.M) continue;
                    if (both[j]) *reinterpret_cast<floatx2u*>(to) = floatx2u{even[i][j][r], acc[i][j][r]};
                    else if (live[j]) *to = even[i][j][r];
                }
    } else finish(std::false_type{}, c, acc, live, 0, n_units);
}

// y = act(sum of the parts + bias): element idx is (image, channel, pixel)
__global__ __launch_bounds__(256) void cl_sum_kernel(float* y, const float* __restrict__ partial, const float* bias, unsigned total, int parts,
                                                     unsigned plane, unsigned M, long sp, long sc, long sn, int relu) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    float s = cl_sum_parts(parts, [&](int q) { return partial[(long)q * total + i]; });
    if (bias) {
        const unsigned pl = i / plane, px = i - pl * plane, img = pl / M, o = pl - img * M;
        s += bias[img * sn + o * sc + px * sp];
    }
    if (relu) s = s > 0.f ? s : 0.f;
    y[i] = s;
}

// ---- weight gradient -------------------------------------------------------------------------------------------------
struct ClDwArgs {
    const _Float16* x;                  // channel-last, padded
    const _Float16* dz;                 // channel-last, pixels of all images one after the other
    float* dw;
    float* partial;                     // [part][dw] bare sums, or null
    int units, cu, Kw, C, taps, O, Op, Os;  // units (tap, 8 channels); per tap; dz channels in whole units, dz row
    int dr, ds;                         // x copy offset between tap rows / columns, elements
    int Ho, Wo, pixels;                 // pixels of the contraction: of all images, or of one with a weight copy per image
    unsigned step_w, step_h;            // x copy offset between output columns / rows, elements
    long x_img;                         // between images
    int adv_h, adv_w;                   // one group's step of 64 KG pixels beyond whole images, as rows and columns
    unsigned adv, wrap_w, wrap_h;       // that step, and what a row's and an image's end add to it, in bytes modulo 2^32
    unsigned x_bytes, z_bytes;
    long z_img, dw_img;                 // elements of one image of dz / of one weight copy
    long total;                         // elements of dw
    int parts, part_steps, tiles_m, tiles;
    ClDiv by_cu, by_kw, by_hw, by_w, by_tiles_m;
};

// 64 TM rows (8 TM units) x 64 TN output channels per workgroup, contraction over steps of 64 pixels. In LDS a row is a pixel: 64
// channels of x at one tap (or of dz), so the MFMA fragments, which want 8 pixels of one channel, are read with the transposing
// LDS load: 16 lanes read 4 pixels x 16 channels and each gets 4 pixels of one channel. Swizzle and ring as above. A pixel past
// the end is zeros in both operands (an offset outside the buffer), so nothing of a neighbour enters a sum.
template <typename T>
__global__ __launch_bounds__(T::THREADS, 2) void cl_dw_kernel(const ClDwArgs p) {
    constexpr int TM = T::TM, TN = T::TN, KG = T::KG, NST = T::NST, STAGE = T::STAGE;
    constexpr int MT = T::BM / 64, NT = T::BN / 64, Q = 4 / T::WN, LOADS = Q * (MT + NT);     // 64-channel tiles; groups of 8 pixels per wave and step
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & (2 * T::WN - 1), kg = KG > 1 ? __builtin_amdgcn_readfirstlane(tid / T::GROUP) : 0;
    const int wm = wave / T::WN, wn = wave % T::WN, li = lane & 31, lh = lane >> 5;
    const int lin = cl_xcd_place(blockIdx.x, p.tiles);
    const int tile_n = cl_quot(lin, p.by_tiles_m), tile_m = lin - tile_n * p.tiles_m;
    const int z = blockIdx.z;
    const int4_t rx = cl_buffer(p.x + z * p.x_img, p.x_bytes), rz = cl_buffer(p.dz + z * p.z_img, p.z_bytes);

    // offsets of this lane's units, for each of its groups of 8 pixels (the unit in a slot differs between even and odd groups)
    const int ch = (lane & 7) ^ (lane >> 4);
    unsigned off_x[MT][Q], off_z[NT][Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int c = ch ^ (((wave * Q + q) & 1) * 4);
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const int u = (tile_m * MT + t) * 8 + c, tap = cl_quot(u, p.by_cu), r = cl_quot(tap, p.by_kw), s = tap - r * p.Kw;
            off_x[t][q] = u < p.units ? (unsigned)(r * p.dr + s * p.ds + (u - tap * p.cu) * 8) * 2u : CL_OUT;
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int o = ((tile_n * NT + t) * 8 + c) * 8;
            off_z[t][q] = o < p.Op ? (unsigned)o * 2u : CL_OUT;
        }
    }
    // the pixels this lane loads per step, walked from step to step
    const int step0 = blockIdx.y * p.part_steps, last = step0 + p.part_steps, all = (p.pixels + 63) / 64;
    const int n_steps = (last < all ? last : all) - step0, steps = (n_steps + KG - 1) / KG;
    const int limit = (step0 + n_steps) * 64 < p.pixels ? (step0 + n_steps) * 64 : p.pixels;
    int px[Q], row[Q], col[Q];
    unsigned at[Q];                                                  // bytes
#pragma unroll
    for (int q = 0; q < Q; q++) {
        px[q] = (step0 + kg) * 64 + (wave * Q + q) * 8 + (lane >> 3);
        const int hw = p.Ho * p.Wo, img = cl_quot(px[q], p.by_hw), r = px[q] - img * hw;
        row[q] = cl_quot(r, p.by_w);
        col[q] = r - row[q] * p.Wo;
        at[q] = (img * (unsigned)p.x_img + row[q] * p.step_h + col[q] * p.step_w) * 2u;
    }
    char* ring = lds + kg * NST * STAGE;
    const unsigned ring_at = cl_lds(ring) + wave * Q * 1024;
    auto request = [&](int slot) {
        const unsigned sa = ring_at + slot * STAGE;
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const bool in = px[q] < limit;
            const unsigned bx = at[q], bz = (unsigned)px[q] * (unsigned)p.Os * 2u;
#pragma unroll
            for (int t = 0; t < MT; t++) cl_load(rx, sa + t * 8192 + q * 1024, in ? bx + off_x[t][q] : CL_OUT);
#pragma unroll
            for (int t = 0; t < NT; t++) cl_load(rz, sa + (MT + t) * 8192 + q * 1024, in ? bz + off_z[t][q] : CL_OUT);
        }
    };
    auto advance = [&]() {
#pragma unroll
        for (int q = 0; q < Q; q++) {
            px[q] += 64 * KG;
            col[q] += p.adv_w; row[q] += p.adv_h;
            at[q] += p.adv;
            if (col[q] >= p.Wo) { col[q] -= p.Wo; row[q]++; at[q] += p.wrap_w; }
            if (row[q] >= p.Ho) { row[q] -= p.Ho; at[q] += p.wrap_h; }
        }
    };

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    // fragment addresses: group of 16 lanes g takes channels (g & 1) * 16 .. + 15 and pixels (g >> 1) * 8 + h * 4 .. + 3 of a k16 step
    const int g = lane >> 4, i4 = lane & 15;
    int frag[2][2];                                                  // [half of the 8 pixels][32-channel block]
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int f = 0; f < 2; f++) {
            const int r = (g >> 1) * 8 + h * 4 + (i4 >> 2), chunk = f * 4 + (g & 1) * 2 + ((i4 & 3) >> 1);
            frag[h][f] = r * 128 + ((chunk ^ ((r >> 1) & 7)) << 4) + (i4 & 1) * 8;
        }
    auto read = [&](const char* base, int block, int k16) {         // block: 32-channel block of the operand's tiles
        const char* t = base + (block >> 1) * 8192 + k16 * 2048;
        return cl_read_turned(t + frag[0][block & 1], t + frag[1][block & 1]);
    };

    for (int t = 0; t < NST - 1; t++) {
        request(t);
        advance();
    }
    ClSums<TM, TN> sums;
    const int chain = cl_chain(steps);
    int slot = 0;
    for (int t = 0; t < steps; t++) {
        cl_wait_vmcnt<(NST - 2) * LOADS>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        request(slot == 0 ? NST - 1 : slot - 1);
        const char* base = ring + slot * STAGE;
        half8_t af[4][TM], bf[4][TN];
#pragma unroll
        for (int k = 0; k < 4; k++) {
#pragma unroll
            for (int i = 0; i < TM; i++) af[k][i] = read(base, wm * TM + i, k);
#pragma unroll
            for (int j = 0; j < TN; j++) bf[k][j] = read(base + MT * 8192, wn * TN + j, k);
            __builtin_amdgcn_sched_barrier(0);                      // in the order of their use
        }
        advance();                                                  // in the time the reads take
        sums.take(acc, t, chain);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[k][i], bf[k][j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        slot = slot == NST - 1 ? 0 : slot + 1;
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

    // lane = output channel, registers = (unit r >> 2, channel lh * 4 + (r & 3))
    const bool split = p.parts > 1;
    float* dst = (split ? p.partial + blockIdx.y * p.total : p.dw) + z * p.dw_img;
    int where[TM][16];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int u = tile_m * MT * 8 + (wm * TM + i) * 4 + q, tap = cl_quot(u, p.by_cu), c0 = (u - tap * p.cu) * 8 + lh * 4;
#pragma unroll
            for (int e = 0; e < 4; e++) where[i][q * 4 + e] = u < p.units && c0 + e < p.C ? ((c0 + e) * p.taps + tap) * p.O : -1;
        }
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int o = tile_n * T::BN + (wn * TN + j) * 32 + li;
        const bool live = o < p.O;
        if (!split) {                                               // dw += : all of a lane's old values before its first store
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += live && where[i][r] >= 0 ? dst[where[i][r] + o] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (live && where[i][r] >= 0) dst[where[i][r] + o] = acc[i][j][r];
    }
}

// ---- host side ----------------------------------------------------------------------------------------------------------

struct ClPlan { int tile, parts; };                                 // tile: index into the list of cl_pick
struct ClTileShape { int bm, bn, kg; };
constexpr ClTileShape CL_TILES[] = {{64, 64, 1}, {64, 64, 2}, {128, 64, 1}, {64, 128, 1}, {128, 128, 1}};
template <typename F>
static int cl_pick(int tile, F go) {
    switch (tile) {
        case 0: return go(ClTile<1, 1, 2, 1>{});
        case 1: return go(ClTile<1, 1, 2, 2>{});
        case 2: return go(ClTile<2, 1, 2, 1>{});
        case 3: return go(ClTile<1, 2, 2, 1>{});
        default: return go(ClTile<2, 1, 4, 1>{});
    }
}
// How a product is cut: `list` workgroup tiles of each kind (CL_TILES) for one weight copy, `steps` k steps of 8 units or 64 pixels in
// the longest sum, `after` in the other sum of its workgroup (columns in pairs) and `mean` in both on average (the classes of a data gradient
// differ), `copies` weight copies, `out` bytes of result.
struct ClWork {
    long dw, tiles[5], copies, steps, after, paired;
    double mean, prep, out;             // prep: bytes the first launch moves
};

// Estimated time in us, and the plan it is for. Measured on 249 (layer, direction) pairs with 15 plans each (layers of 1 to 32 images, 3 to 512
// channels, 7 x 7 to 224 x 224, kernels 3, 5 and 7, strides 1 and 2) and fitted: the plan chosen is 1.3 % slower than the best of the 15
// in the geometric mean, 16 % at worst. A k step of a workgroup alone on its CU takes `alone`, of two that share one `pair` together.
static double cl_plan_search(const ClWork& w, ClPlan& best) {
    static const double alone[2][5] = {{0.191, 0.295, 0.346, 0.423, 0.484}, {0.358, 0.515, 0.493, 0.468, 0.575}};
    static const double pair[2][5] = {{0.375, 0.360, 0.579, 0.461, 0.500}, {0.441, 0.560, 0.633, 0.427, 0.600}};
    static const double first[5] = {4.2, 5.1, 4.2, 4.2, 4.8};        // launch, first request and result of a workgroup
    static const int cuts[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};
    const double cus = device_cu_count();
    double least = 1e30;
    for (int t = 0; t < 5; t++) {
        const int kg = CL_TILES[t].kg;
        // pairs on 128 x 64, a weight copy per image (16 x 352 x 26 x 26 <- 38 7x7 50.9 us, 41.6 on 64 x 128; shared, 16 x 80 x 49 x 49 <- 87 34.3, 38.9)
        const double slow = w.paired && t == 2 && w.copies > 1 ? 1.2 : 1.0;
        for (int cut : cuts) {
            if (cut > 1 && (cut > w.steps || (double)cut * w.out > 5e8 || (double)w.tiles[t] * w.copies * cut > 8.0 * cus)) break;
            // each sum is cut at the same steps, so the first part has most of both
            const long per = (w.steps + cut - 1) / cut, parts = (w.steps + per - 1) / per, also = w.after < per ? w.after : per, own = (per + kg - 1) / kg + (also + kg - 1) / kg;
            if (cut > 1 && parts != cut) continue;
            const bool two = t != 1 && t != 4 && (w.dw || (per + also) * 8 <= (t == 0 ? 1900 : 900));      // LDS for two: ring and table
            const double wgs = (double)w.tiles[t] * w.copies * parts, load = w.mean / parts / kg;
            double main = first[t];
            if (wgs <= cus) main += own * alone[w.dw][t] * slow;
            else {
                const double rounds = wgs / (cus * (two ? 2 : 1)), filled = rounds < 1.0 ? 1.0 : rounds < 3.0 ? std::ceil(rounds) : rounds + 0.4;
                const double share = wgs / cus - 1.0 < 1.0 ? wgs / cus - 1.0 : 1.0;
                const double step = two ? alone[w.dw][t] + (pair[w.dw][t] - alone[w.dw][t]) * share : alone[w.dw][t];
                main += filled * (rounds > 1.0 ? load : (double)own) * step * slow + (filled - 1.0) * 2.7;
            }
            main += w.out / (w.paired ? 5.5e6 : 3.3e6);               // stores of 8 bytes a lane, of 4
            if (parts > 1) main += 2.6 + w.out * (2.0 * parts + 1.0) / 9.2e6;
            if (main < least) {
                least = main;
                best = ClPlan{t, (int)parts};
            }
        }
    }
    return 3.9 + w.prep / 5e6 + least;
}
static double cl_plan(const ClWork& w, ClPlan& best) {
    struct Found { ClPlan plan; double cost; };
    struct Key { ClWork w; long cus; };
    static thread_local PlanCache<Key, Found> cache;
    bool known;
    Found& f = cache.at(Key{w, device_cu_count()}, known);
    if (!known) f.cost = cl_plan_search(w, f.plan);
    best = f.plan;
    return f.cost;
}
// read per call (tests, benchmarking): "tile,parts"
static void plan_env(ClPlan& pl) {
    const char* e = getenv("NZHIP_CONV_CL_PLAN");
    ClPlan q;
    if (e && sscanf(e, "%d,%d", &q.tile, &q.parts) == 2 && q.tile >= 0 && q.tile < 5 && q.parts >= 1) pl = q;
}

template <typename K, typename A>
static int launch(K kfn, dim3 grid, int threads, size_t lds, const A& a, hipStream_t s, const char* what) {
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kfn), (int)lds, what)) return rc;
    hipLaunchKernelGGL(kfn, grid, dim3((unsigned)threads), lds, s, a);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? NZHIP_OK : set_hip_error(e, what);
}

static ClWork conv_work(const ClArgs& a, int copies, double prep) {
    ClWork w = {};
    w.copies = copies; w.prep = prep; w.out = (double)a.y_total * 4.0;
    w.paired = a.paired;
    for (int t = 0; t < 5; t++) {
        double all = 0.0;
        for (int i = 0; i < a.n_classes; i += a.paired ? 2 : 1) {
            const ClClass& c = a.cls[i];
            const long n = (((long)a.images * c.Hc * c.Wc + CL_TILES[t].bn - 1) / CL_TILES[t].bn) * ((a.M + CL_TILES[t].bm - 1) / CL_TILES[t].bm);
            const long k = ((long)c.nr * c.ns * a.cu + 7) / 8, k2 = a.paired ? ((long)a.cls[i + 1].nr * a.cls[i + 1].ns * a.cu + 7) / 8 : 0;
            w.tiles[t] += n;
            all += (double)n * (double)(k + k2);
            if (k + k2 > w.steps + w.after) {
                w.steps = std::max(k, k2);
                w.after = std::min(k, k2);
            }
        }
        if (t == 0) w.mean = w.tiles[0] ? all / (double)w.tiles[0] : 0.0;
    }
    if (w.steps < 1) w.steps = 1;
    return w;
}

// Tiles and parts of a product; a.M, a.cls (taps and pixels) and everything else but the addresses is set. Bytes of its partial sums.
static size_t conv_cut(ClArgs& a, int copies, ClPlan& pl) {
    int units = 0;
    for (int i = 0; i < a.n_classes; i++) {
        const int u = a.cls[i].nr * a.cls[i].ns * a.cu;
        if (u > units) units = u;
    }
    const int steps = (units + 7) / 8;
    cl_plan(conv_work(a, copies, 0.0), pl);
    plan_env(pl);
    const ClTileShape sh = CL_TILES[pl.tile];
    a.units = units;
    a.part_units = ((steps + pl.parts - 1) / pl.parts) * 8;
    if (a.part_units < 8) a.part_units = 8;
    a.parts = (units + a.part_units - 1) / a.part_units;
    if (a.parts < 1) a.parts = 1;
    a.tiles_m = (a.M + sh.bm - 1) / sh.bm;
    int most = 0;
    a.by_cu = cl_div(a.cu); a.by_tiles_m = cl_div(a.tiles_m);
    for (int i = 0; i < a.n_classes; i++) {
        ClClass& c = a.cls[i];
        c.by_ns = cl_div(c.ns ? c.ns : 1); c.by_hw = cl_div(c.Hc * c.Wc); c.by_w = cl_div(c.Wc);
        const int tiles = (int)(((long)a.images * c.Hc * c.Wc + sh.bn - 1) / sh.bn) * a.tiles_m;
        if (tiles > most) most = tiles;
    }
    const int groups = a.paired ? a.n_classes / 2 : a.n_classes;
    a.tiles = most * groups;
    a.by_groups = cl_div(groups);
    return a.parts > 1 ? (size_t)a.parts * a.y_total * sizeof(float) : 0;
}

// its launches, operands and partial sums in place
static int conv_product(const ClArgs& a, int copies, const ClPlan& pl, hipStream_t s) {
    const dim3 grid((unsigned)a.tiles, (unsigned)a.parts, (unsigned)copies);
    const int mu = a.part_units < a.units ? a.part_units : a.units, kgs = CL_TILES[pl.tile].kg;
    size_t steps = 0;                                                 // of one workgroup's sum or two, at most
    for (int i = 0; i < a.n_classes; i += a.paired ? 2 : 1) {
        size_t n = 0;
        for (int k = i; k < i + (a.paired ? 2 : 1); k++) n += ((std::min(a.cls[k].nr * a.cls[k].ns * a.cu, mu) + 7) / 8 + kgs - 1) / kgs;
        steps = std::max(steps, n);
    }
    const size_t table = (steps + 4) * kgs * 8 * sizeof(int2);       // and the ring's stages
    if (gemm_trace())
        fprintf(stderr, "nzhip_conv: channel-last copies, tile %d, %d part(s), planned %d%s\n", pl.tile, a.parts, pl.parts, a.paired ? ", columns in pairs" : "");
    int rc;
    auto go = [&](auto tile) {
        using T = decltype(tile);
        return launch(a.paired          ? cl_conv_kernel<T, true, true, true>
                      : a.n_classes > 1 ? cl_conv_kernel<T, true, true, false>
                      : a.dy_h          ? cl_conv_kernel<T, true, false, false>
                                        : cl_conv_kernel<T, false, false, false>, grid, T::THREADS, T::RING + table, a, s, "cl_conv kernel launch");
    };
    rc = cl_pick(pl.tile, go);
    if (rc == NZHIP_OK && a.parts > 1) {
        hipLaunchKernelGGL(cl_sum_kernel, dim3((unsigned)((a.y_total + 255) / 256)), dim3(256), 0, s, a.y, a.partial, a.bias, (unsigned)a.y_total, a.parts,
                           (unsigned)a.plane, (unsigned)a.M, a.bias_sp, a.bias_sc, a.bias_sn, a.relu);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) rc = set_hip_error(e, "cl_sum kernel launch");
    }
    return rc;
}

// The extents the kernels' 32-bit offsets and tables hold: copies and result below 2 GiB, a unit table beside the largest ring.
// 0: not, 1: yes, 2: yes and to be taken whatever the layer.
int cl_conv_fits(ClDirection dir, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w, size_t stride, size_t pad, size_t w_batch) {
    if (!N || !C || !O || !H || !W || (dir == CL_DATA && stride > 3) || K_h > 64 || K_w > 64 || H > 16384 || W > 16384 || pad > 64 || stride > 64 || C > 65535 || O > 65535 || N > 32768) return 0;
    const size_t taps = K_h * K_w, Cp = (C + 7) / 8 * 8, Op = (O + 7) / 8 * 8, Cs = C + 128, Os = O + 128, Hp = H + 2 * pad + K_h, Wp = W + 2 * pad + K_w, lim = 1u << 30;
    if (!(N * Hp * Wp * Cs < lim && N * Hp * Wp * Os < lim && w_batch * (taps * Cp + 128) * O < lim && w_batch * (taps * Op + 128) * C < lim &&
           N * (H + 2 * pad) * (W + 2 * pad) * (C > O ? C : O) < lim / 2 && w_batch * taps * C * O < lim && taps * Cp / 8 <= 3500 && taps * Op / 8 <= 3500)) return 0;
    const char* env = getenv("NZHIP_CONV_CL");                       // read per call (tests, benchmarking): 0 never, 1 wherever they fit
    return env ? (atoi(env) ? 2 : 0) : 1;
}

// the product of a forward, of a data gradient: everything but the operands' addresses. Zero rows and columns around dy: edge[0..3]
static void forward_args(ClArgs& a, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w, size_t stride, size_t pad, size_t w_batch) {
    const int Ho = (int)((H + 2 * pad - K_h) / stride + 1), Wo = (int)((W + 2 * pad - K_w) / stride + 1);
    const int Cp = round8((int)C), taps = (int)(K_h * K_w), Hp = (int)(H + 2 * pad), Wp = (int)(W + 2 * pad);
    const int Cs = cl_pitch((int)C);
    a.M = (int)O; a.w_row = cl_pitch(taps * Cp); a.cu = Cp / 8; a.Kw = (int)K_w;
    a.step_h = (int)stride * Wp * Cs; a.step_w = (int)stride * Cs;
    a.images = w_batch > 1 ? 1 : (int)N;
    a.x_img = (long)Hp * Wp * Cs; a.w_img = (long)O * a.w_row; a.y_img = (long)O * Ho * Wo;
    a.w_bytes = (unsigned)(a.w_img * 2); a.x_bytes = (unsigned)(a.images * a.x_img * 2);
    a.plane = (long)Ho * Wo; a.y_total = (long)N * a.y_img;
    a.n_classes = 1;
    a.cls[0] = {(int)K_h, (int)K_w, 0, 1, 0, 1, Wp * Cs, Cs, Ho, Wo, 0, 0, Wo, 1, 0, 0, {}, {}, {}};
}

static void data_args(ClArgs& a, int (&edge)[4], size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w, size_t stride, size_t pad,
                      size_t w_batch) {
    // dx[n][c][h][w] (+)= sum over (tap, o) of w[(c, tap)][o] dy[n][o][(h + pad - r) / stride][(w + pad - s) / stride], the taps with whole
    // quotients: for the elements whose h + pad is i modulo the stride, rows r = i + k stride of the kernel and row h' - k of dy.
    const int Ho = (int)((H + 2 * pad - K_h) / stride + 1), Wo = (int)((W + 2 * pad - K_w) / stride + 1), st = (int)stride;
    const int Op = round8((int)O), taps = (int)(K_h * K_w);
    struct Side { int lo, n, t; };                                                // h' from lo on, how many, and the taps
    auto side = [&](int i, int extent, int k) {
        Side r;
        r.lo = (int)pad > i ? ((int)pad - i + st - 1) / st : 0;                   // smallest h' with st h' + i - pad >= 0
        const int hi = extent - 1 + (int)pad - i;                                 // st h' <= hi
        r.n = hi < 0 ? 0 : hi / st - r.lo + 1;
        if (r.n < 0) r.n = 0;
        r.t = k > i ? (k - i + st - 1) / st : 0;
        return r;
    };
    for (int& e : edge) e = 0;
    for (int i = 0; i < st; i++) {
        const Side h = side(i, (int)H, (int)K_h), v = side(i, (int)W, (int)K_w);
        if (h.n) { edge[0] = std::max(edge[0], h.t - 1 - h.lo); edge[1] = std::max(edge[1], h.lo + h.n - Ho); }
        if (v.n) { edge[2] = std::max(edge[2], v.t - 1 - v.lo); edge[3] = std::max(edge[3], v.lo + v.n - Wo); }
    }
    const int Hp = Ho + edge[0] + edge[1], Wp = Wo + edge[2] + edge[3];
    const int Os = cl_pitch((int)O);
    a.M = (int)C; a.w_row = cl_pitch(taps * Op); a.cu = Op / 8; a.Kw = (int)K_w; a.dy_h = Ho; a.dy_w = Wo;
    a.step_h = Wp * Os; a.step_w = Os;
    a.images = w_batch > 1 ? 1 : (int)N;
    a.x_img = (long)Hp * Wp * Os; a.w_img = (long)C * a.w_row; a.y_img = (long)C * H * W;
    a.w_bytes = (unsigned)(a.w_img * 2); a.x_bytes = (unsigned)(a.images * a.x_img * 2);
    a.plane = (long)H * W; a.y_total = (long)N * a.y_img;
    const bool pairs = st == 2 && W > 1;                            // columns 0, 2, .. first
    for (int i = 0; i < st; i++)
        for (int q = 0; q < st; q++) {
            const int j = pairs ? (q + (int)pad) & 1 : q;
            const Side h = side(i, (int)H, (int)K_h), v = side(j, (int)W, (int)K_w);
            if (!h.n || !v.n) continue;
            a.cls[a.n_classes++] = {h.t, v.t, i, st, j, st, -Wp * Os, -Os, h.n, v.n, ((h.lo + edge[0]) * Wp + v.lo + edge[2]) * Os,
                                    (st * h.lo + i - (int)pad) * (int)W + st * v.lo + j - (int)pad, st * (int)W, st, h.lo, v.lo, {}, {}, {}};
        }
}

int cl_conv_forward(float* y, const float* x, const float* w, const float* bias, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h,
                    size_t K_w, size_t stride, size_t pad, size_t w_batch, int64_t bias_sp, int64_t bias_sc, int64_t bias_sn, int relu, bool may_keep, hipStream_t s) {
    ClArgs a = {};
    forward_args(a, N, C, H, W, O, K_h, K_w, stride, pad, w_batch);
    const int Cp = round8((int)C), taps = (int)(K_h * K_w);
    _Float16* xc = nullptr;
    if (int rc = workspace_alloc(reinterpret_cast<void**>(&xc), N * (size_t)a.x_img * 2, s)) return rc;
    ImageLease lease;
    const uint64_t key[PREPARED_KEY_WORDS] = {0xC1u | (uint64_t)K_h << 8 | (uint64_t)K_w << 16, reinterpret_cast<uintptr_t>(w), C, O, 0, 0, w_batch};
    int rc = may_keep ? image_acquire(PREPARED_CONV_W, key, w_batch * (size_t)a.w_img * 2, s, &lease)
                      : workspace_alloc(&lease.ptr, w_batch * (size_t)a.w_img * 2, s);
    if (rc) {
        workspace_free(xc, s);
        return rc;
    }
    const int copies = w_batch > 1 ? (int)N : 1;
    ClPlan pl = {0, 1};
    if (const size_t bytes = conv_cut(a, copies, pl)) rc = workspace_alloc(reinterpret_cast<void**>(&a.partial), bytes, s);
    if (rc) {
        may_keep ? image_release(lease, s, false) : workspace_free(lease.ptr, s);
        workspace_free(xc, s);
        return rc;
    }
    ClPrepArgs pa = {};
    prep_planes(pa.job[0], x, xc, (long)N, (int)C, Cp, (int)H, (int)W, (int)(H + 2 * pad), (int)(W + 2 * pad), (int)pad, (int)pad);
    if (lease.fill) prep_weights(pa.job[1], w, reinterpret_cast<_Float16*>(lease.ptr), (long)w_batch, (int)C, Cp, taps, (int)O);
    rc = prep_launch(pa, s);
    const bool enqueued = rc == NZHIP_OK;
    if (rc == NZHIP_OK) {
        a.w = reinterpret_cast<const _Float16*>(lease.ptr); a.x = xc; a.y = y; a.bias = bias;
        a.bias_sp = bias_sp; a.bias_sc = bias_sc; a.bias_sn = bias_sn; a.relu = relu;
        a.early_bias = bias && a.parts == 1 && (long)a.tiles * copies <= 2 * device_cu_count();
        rc = conv_product(a, copies, pl, s);
    }
    const int rc2 = may_keep ? image_release(lease, s, enqueued) : workspace_free(lease.ptr, s), rc3 = workspace_free(xc, s);
    const int rc4 = a.partial ? workspace_free(a.partial, s) : NZHIP_OK;
    return rc ? rc : rc2 ? rc2 : rc3 ? rc3 : rc4;
}

// Whether a data gradient at stride 2 computes neighbouring columns in one workgroup. One class of columns after the other stores every second 4 bytes
// of a line, twice: 16 x 128 x 56 x 56 <- 128 15 of 22 us, 2.3 TB/s. In pairs 8 bytes a lane go out at 5 TB/s, by half as many workgroups with sums twice
// as long, which layers of few tiles do not fill the chip with. The model has both; on 744 layers the way it takes at this margin is
// 0.7 % behind the better one in the geometric mean. 204 go in pairs, three of them 7 to 9 % slower so (16 x 288 x 19 x 19 <- 180 24.9 or 27.2 us, a weight copy per
// image); not taken though ahead are 34 by more than 5 %, most of all long sums on small images (16 x 508 x 16 x 16 <- 318 7x7 57.9 or 44.5, 4 x 32 x 80 x 80 <- 480 25.8 or
// 21.7). 16 x 128 x 56 x 56 <- 128 30.5 -> 25.4 us, 16 x 64 x 128 x 128 <- 128 51 -> 42, 8 x 392 x 80 x 80 <- 16 41 -> 25, 4 x 320 x 160 x 160 <- 30 68 -> 38.
// Where the stores would gain less than 1.2 % the model's last rounds decide, and not well (10 x 13 x 92 x 92 <- 389 7x7 120 or 124).
// Not taken: 16 x 17 x 27 x 27 <- 128 7x7 15.5 or 20.9, 10 x 39 x 32 x 32 <- 240 12.8 or 15.6.
static bool cl_paired(const ClArgs& a, size_t N, size_t H, size_t W, size_t K_h, size_t pad, size_t stride, int copies) {
    if (stride != 2 || W < 2) return false;
    if (const char* e = getenv("NZHIP_CONV_CL_PAIRED")) return atoi(e);      // read per call (tests, benchmarking)
    struct Key { long N, C, H, W, cu, K_h, K_w, pad, copies, cus; };
    struct Found { bool paired; };
    static thread_local PlanCache<Key, Found> cache;
    bool known;
    Found& f = cache.at(Key{(long)N, a.M, (long)H, (long)W, a.cu, (long)K_h, a.Kw, (long)pad, copies, device_cu_count()}, known);
    if (!known) {
        ClPlan pl;
        ClArgs two = a;
        const double one = cl_plan(conv_work(a, copies, 0.0), pl);
        two.paired = 1;
        f.paired = 1.1 * cl_plan(conv_work(two, copies, 0.0), pl) < one && (double)a.y_total * 5e-7 > 0.012 * one;      // that the stores gain
    }
    return f.paired;
}

int cl_conv_backward_data(float* dx, const float* dy, const float* w, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w,
                          size_t stride, size_t pad, size_t w_batch, int accumulate, hipStream_t s) {
    ClArgs a = {};
    int edge[4];
    data_args(a, edge, N, C, H, W, O, K_h, K_w, stride, pad, w_batch);
    const int Ho = (int)((H + 2 * pad - K_h) / stride + 1), Wo = (int)((W + 2 * pad - K_w) / stride + 1), Op = round8((int)O);
    _Float16* zc = nullptr;
    _Float16* wc = nullptr;
    if (int rc = workspace_alloc(reinterpret_cast<void**>(&zc), N * (size_t)a.x_img * 2, s)) return rc;
    const int copies = w_batch > 1 ? (int)N : 1;
    a.paired = cl_paired(a, N, H, W, K_h, pad, stride, copies);
    ClPlan pl = {0, 1};
    int rc = workspace_alloc(reinterpret_cast<void**>(&wc), w_batch * (size_t)a.w_img * 2, s);
    if (const size_t bytes = rc ? 0 : conv_cut(a, copies, pl)) rc = workspace_alloc(reinterpret_cast<void**>(&a.partial), bytes, s);
    if (rc) {
        if (wc) workspace_free(wc, s);
        workspace_free(zc, s);
        return rc;
    }
    ClPrepArgs pa = {};
    prep_planes(pa.job[0], dy, zc, (long)N, (int)O, Op, Ho, Wo, Ho + edge[0] + edge[1], Wo + edge[2] + edge[3], edge[0], edge[2]);
    prep_rows(pa.job[1], w, wc, (long)(w_batch * C * K_h * K_w), (int)(K_h * K_w), (int)O, Op);
    rc = prep_launch(pa, s);
    if (rc == NZHIP_OK) {
        a.w = wc; a.x = zc; a.y = dx;
        if (accumulate) { a.bias = dx; a.bias_sp = 1; a.bias_sc = a.plane; a.bias_sn = a.y_img; }
        rc = conv_product(a, copies, pl, s);
    }
    const int rc2 = workspace_free(wc, s), rc3 = workspace_free(zc, s), rc4 = a.partial ? workspace_free(a.partial, s) : NZHIP_OK;
    return rc ? rc : rc2 ? rc2 : rc3 ? rc3 : rc4;
}

static ClWork dw_work(size_t N, size_t C, size_t O, size_t taps, size_t P, size_t w_batch) {
    ClWork w = {};
    const long rows = (long)(taps * ((C + 7) / 8) * 8), pixels = (long)((w_batch > 1 ? 1 : N) * P);
    w.dw = 1;
    w.copies = w_batch > 1 ? (int)N : 1;
    for (int t = 0; t < 5; t++) w.tiles[t] = ((rows + CL_TILES[t].bm - 1) / CL_TILES[t].bm) * (((long)O + CL_TILES[t].bn - 1) / CL_TILES[t].bn);
    w.steps = (pixels + 63) / 64;
    w.mean = (double)w.steps;
    w.out = 8.0 * (double)w_batch * (double)(C * taps * O);
    return w;
}

double cl_conv_cost(ClDirection dir, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w, size_t stride, size_t pad, size_t w_batch) {
    const double P = (double)((H + 2 * pad - K_h) / stride + 1) * (double)((W + 2 * pad - K_w) / stride + 1), x = 4.0 * N * C * H * W, y = 4.0 * N * O * P;
    const double weights = 4.0 * w_batch * C * K_h * K_w * O;
    ClPlan pl;
    if (dir == CL_WEIGHTS) {
        ClWork w = dw_work(N, C, O, K_h * K_w, (size_t)P, w_batch);
        w.prep = 1.5 * (x + y);
        return cl_plan(w, pl);
    }
    ClArgs a = {};
    int edge[4];
    if (dir == CL_FORWARD) {
        forward_args(a, N, C, H, W, O, K_h, K_w, stride, pad, w_batch);
    } else {
        data_args(a, edge, N, C, H, W, O, K_h, K_w, stride, pad, w_batch);
        a.paired = C >= 8 && cl_paired(a, N, H, W, K_h, pad, stride, w_batch > 1 ? (int)N : 1);
    }
    return cl_plan(conv_work(a, w_batch > 1 ? (int)N : 1, 1.5 * weights + (dir == CL_FORWARD ? x : y) + 2.0 * N * (double)a.x_img), pl);
}

int cl_conv_backward_weights(float* dw, const float* x, const float* dy, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w,
                             size_t stride, size_t pad, size_t w_batch, hipStream_t s) {
    const int Ho = (int)((H + 2 * pad - K_h) / stride + 1), Wo = (int)((W + 2 * pad - K_w) / stride + 1);
    const int Cp = round8((int)C), Op = round8((int)O), taps = (int)(K_h * K_w), Hp = (int)(H + 2 * pad), Wp = (int)(W + 2 * pad);
    const int Cs = cl_pitch((int)C), Os = cl_pitch((int)O);
    const size_t x_elems = N * Hp * Wp * (size_t)Cs, z_elems = N * Ho * Wo * (size_t)Os;
    _Float16* xc = nullptr;
    if (int rc = workspace_alloc(reinterpret_cast<void**>(&xc), (x_elems + z_elems) * 2, s)) return rc;      // (rows of whole 16 bytes)
    _Float16* zc = xc + x_elems;
    ClDwArgs a = {};
    const int copies = w_batch > 1 ? (int)N : 1, images = w_batch > 1 ? 1 : (int)N;
    a.x = xc; a.dz = zc; a.dw = dw;
    a.cu = Cp / 8; a.units = taps * a.cu; a.Kw = (int)K_w; a.C = (int)C; a.taps = taps; a.O = (int)O; a.Op = Op;
    a.dr = Wp * Cs; a.ds = Cs; a.Os = Os;
    a.Ho = Ho; a.Wo = Wo; a.pixels = images * Ho * Wo;
    a.step_h = (unsigned)(stride * Wp * Cs); a.step_w = (unsigned)(stride * Cs); a.x_img = (long)Hp * Wp * Cs;
    a.z_img = (long)Ho * Wo * Os; a.dw_img = (long)C * taps * O; a.total = copies * a.dw_img;
    a.x_bytes = (unsigned)(images * a.x_img * 2); a.z_bytes = (unsigned)(images * a.z_img * 2);
    ClPlan pl = {0, 1};
    cl_plan(dw_work(N, C, O, taps, (size_t)Ho * Wo, w_batch), pl);
    plan_env(pl);
    const ClTileShape sh = CL_TILES[pl.tile];
    const int adv = 64 * sh.kg, hw = Ho * Wo;
    a.adv_h = adv % hw / Wo; a.adv_w = adv % hw % Wo;
    a.adv = (unsigned)(adv / hw * a.x_img + a.adv_h * (long)a.step_h + a.adv_w * (long)a.step_w) * 2u;
    a.wrap_w = (unsigned)((long)a.step_h - (long)Wo * a.step_w) * 2u;
    a.wrap_h = (unsigned)(a.x_img - (long)Ho * a.step_h) * 2u;
    const int steps = (a.pixels + 63) / 64;
    a.part_steps = (steps + pl.parts - 1) / pl.parts;
    a.parts = (steps + a.part_steps - 1) / a.part_steps;
    a.by_cu = cl_div(a.cu); a.by_kw = cl_div(a.Kw); a.by_hw = cl_div(hw); a.by_w = cl_div(Wo);
    a.tiles_m = (a.units * 8 + sh.bm - 1) / sh.bm;
    a.by_tiles_m = cl_div(a.tiles_m);
    a.tiles = a.tiles_m * (int)((O + sh.bn - 1) / sh.bn);
    float* partial = nullptr;
    if (a.parts > 1)
        if (int rc = workspace_alloc(reinterpret_cast<void**>(&partial), (size_t)a.parts * a.total * sizeof(float), s)) {
            workspace_free(xc, s);
            return rc;
        }
    a.partial = partial;
    ClPrepArgs pa = {};
    prep_planes(pa.job[0], x, xc, (long)N, (int)C, Cp, (int)H, (int)W, Hp, Wp, (int)pad, (int)pad);
    prep_planes(pa.job[1], dy, zc, (long)N, (int)O, Op, Ho, Wo, Ho, Wo, 0, 0);
    int rc = prep_launch(pa, s);
    if (rc == NZHIP_OK) {
        const dim3 grid((unsigned)a.tiles, (unsigned)a.parts, (unsigned)copies);
        auto go = [&](auto tile) {
            using T = decltype(tile);
            return launch(cl_dw_kernel<T>, grid, T::THREADS, T::RING, a, s, "cl_dw kernel launch");
        };
        rc = cl_pick(pl.tile, go);
        if (rc == NZHIP_OK && a.parts > 1) {
            hipLaunchKernelGGL(cl_sum_kernel, dim3((unsigned)((a.total + 255) / 256)), dim3(256), 0, s, dw, partial, dw, (unsigned)a.total, a.parts,
                               (unsigned)a.total, 1u, 1L, 0L, 0L, 0);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) rc = set_hip_error(e, "cl_sum kernel launch");
        }
    }
    const int rc2 = partial ? workspace_free(partial, s) : NZHIP_OK, rc3 = workspace_free(xc, s);
    return rc ? rc : rc2 ? rc2 : rc3;
}

}  // namespace nzhip
