// Convolutions of few tiles in one launch without a workspace: the sliced products (nzhip_gemm_slices.hip) on gathered operands.
//
// A small layer on channel-last copies is two launches, of which the first only rounds, and the column-matrix and strided 1x1 ways are two and
// three; each launch is some 4 us of the host's time and 2 of the GPU's before any work. Here the waves gather fp32 themselves: about
// 130 vector instructions and 32 requests for a chunk of 32 k, which is what bounds it (64 KB per CU in 0.5 us at best, the copies' kernels
// take in half the bytes) and why larger layers stay with the others. us a call, calls queued one behind the other, on the ways before and here:
// 16 x 4 x 10 x 10 -> 25 3x3 7.3 / 4.0, 16 x 147 x 53 x 53 -> 16 1x1 at stride 2 15.3 / 5.3, 32 x 9 x 16 x 16 -> 16 7x7 at stride 2 10.8 / 8.1, 1 x 32 x 80 x 80 -> 11 5x5
// 10.3 / 5.7; gradients 32 x 7 x 18 x 18 <- 93 1x1 14.2 / 4.1, 2 x 16 x 12 x 12 <- 48 3x3 8.2 / 4.9. Requests two or three chunks ahead changed nothing.
#include <hip/hip_runtime.h>

#include <cstdlib>

#include "nzhip_conv_cl.h"
#include "nzhip_internal.h"
#include "nzhip_lds_tiles.h"
#include "nzhip_pieces.h"
#include "nzhip_slices.h"

namespace nzhip {

struct ConvSliceArgs {
    const float* w;
    const float* x;                     // what is gathered: x, or dy in a data gradient
    float* y;
    const float* bias;
    const _Float16* image;              // of a forward's weights, kept by the caller: [copy][unit][M, in whole tiles][16 channels]
    int M, K, taps, K_w;                // result channels, contraction channels
    int Hx, Wx, Hr, Wr;                 // planes of the gathered tensor and of the result
    int stride, pad, units, tiles_m, tiles, total, relu, accumulate;      // units: 16 channels of one tap
    unsigned x_bytes, w_bytes;          // of one image, of one weight copy
    long x_img, w_img, y_img, image_img, bias_sp, bias_sc, bias_sn;
    ClDiv by_blocks, by_kw, by_tiles, by_tiles_m, by_wr, by_stride;
};

// where tap (r, s) of a result pixel reads, -1: outside (DATA: or between the pixels of a stride)
template <bool DATA>
__device__ __forceinline__ int slice_tap(const ConvSliceArgs& p, int h0, int w0, int r, int s) {
    int h = DATA ? h0 - r : h0 + r, w = DATA ? w0 - s : w0 + s;
    bool in = true;
    if (DATA && p.stride > 1) {
        const int hq = cl_quot(h < 0 ? 0 : h, p.by_stride), wq = cl_quot(w < 0 ? 0 : w, p.by_stride);
        in = h >= 0 && w >= 0 && hq * p.stride == h && wq * p.stride == w;
        h = hq;
        w = wq;
    }
    return in && (unsigned)h < (unsigned)p.Hx && (unsigned)w < (unsigned)p.Wx ? h * p.Wx + w : -1;
}

// One element of a data gradient, taps outside dy left out: the zeros in their place are no terms of the sum, and times an infinite weight
// they are not nothing either.
__device__ __forceinline__ float slice_terms(const ConvSliceArgs& p, const float* x, const float* w, int h0, int w0, int m) {
    float sum = 0.f;
#pragma unroll 1
    for (int t = 0; t < p.taps; t++) {
        const int r = cl_quot(t, p.by_kw), at = slice_tap<true>(p, h0, w0, r, t - r * p.K_w);
        if (at < 0) continue;
#pragma unroll 1
        for (int k = 0; k < p.K; k++)
            sum = __builtin_fmaf((float)(_Float16)w[(long)(m * p.taps + t) * p.K + k], (float)(_Float16)x[(long)k * p.Hx * p.Wx + at], sum);
    }
    return sum;
}

// 32 result channels x 32 pixels of one image per workgroup, chunks of two units (16 channels of one tap each) dealt to the NW waves. Lanes are the
// pixels: a unit's 16 channels of a pixel are 16 planes apart, 32 lanes read 128 bytes of each. Channels past the last are past the image's end, taps
// outside a plane an offset past any: zeros. Forward weights lie across k the same way (w[(c, tap)][o]); those of a data gradient lie along it. IMAGE: a
// forward whose weights were rounded once, in the order of the fragments; the sums are the same.
template <bool DATA, bool IMAGE, int NW>
__global__ __launch_bounds__(NW * 64, 4) void conv_slices_kernel(const ConvSliceArgs p) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 31, lh = lane >> 5;
    const int lin = cl_xcd_place(blockIdx.x, p.total);
    const int img = cl_quot(lin, p.by_tiles), t = lin - img * p.tiles, tile_p = cl_quot(t, p.by_tiles_m), m0 = (t - tile_p * p.tiles_m) * 32;
    const int pixels = p.Hr * p.Wr, px = tile_p * 32 + li, pc = px < pixels ? px : pixels - 1, i = cl_quot(pc, p.by_wr), j = pc - i * p.Wr;
    const int h0 = DATA ? i + p.pad : i * p.stride - p.pad, w0 = DATA ? j + p.pad : j * p.stride - p.pad;
    const float *xi = p.x + img * p.x_img, *wi = p.w + img * p.w_img;
    const __amdgpu_buffer_rsrc_t rx = slice_buffer(xi, p.x_bytes);
    const __amdgpu_buffer_rsrc_t rw = IMAGE ? slice_buffer(reinterpret_cast<const float*>(p.image + img * p.image_img), (unsigned)(p.units * p.tiles_m) * 1024u) : slice_buffer(wi, p.w_bytes);
    const unsigned plane = (unsigned)(p.Hx * p.Wx) * 4u;
    char* own = lds + wave * 32 * SLICE_PITCH;

    // weights: forward, this lane's output channel; data gradient, the rows this lane loads for all
    unsigned row[4];
    if (DATA) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int m = m0 + q * 8 + (lane >> 3);
            row[q] = (unsigned)((m < p.M ? m : p.M - 1) * p.taps * p.K) * 4u;
        }
    } else {
        row[0] = IMAGE ? (unsigned)((m0 + li) * 2 + lh) * 16u : (unsigned)(m0 + li < p.M ? m0 + li : p.M - 1) * 4u;
    }
    const unsigned w_step = (unsigned)(p.taps * p.M) * 4u;           // forward: from one channel to the next
    const int blocks = (p.K + 15) >> 4;

    struct Chunk {
        unsigned xv[16], wf[DATA || IMAGE ? 1 : 16];
        uint4_t wd[DATA ? 4 : IMAGE ? 2 : 1];
    };
    auto load = [&](Chunk& k, int c) {
        unsigned at_w[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int unit = c * 2 + u, tap = cl_quot(unit, p.by_blocks), b = unit - tap * blocks, r = cl_quot(tap, p.by_kw), s = tap - r * p.K_w;
            const bool any = unit < p.units;
            const int at = any ? slice_tap<DATA>(p, h0, w0, r, s) : -1;
            unsigned o = at >= 0 ? (unsigned)at * 4u + (unsigned)(b * 16 + lh * 8) * plane : CL_OUT;
            asm volatile("" : "+v"(o));
#pragma unroll
            for (int e = 0; e < 8; e++) {
                k.xv[u * 8 + e] = __builtin_amdgcn_raw_buffer_load_b32(rx, o, 0, 0);
                o += plane;
            }
            if (IMAGE) {
                k.wd[u] = __builtin_amdgcn_raw_buffer_load_b128(rw, any ? (unsigned)(unit * p.tiles_m) * 1024u + row[0] : CL_OUT, 0, 0);
            } else if (DATA) {
                at_w[u] = any ? (unsigned)(tap * p.K + b * 16) * 4u : CL_OUT;
            } else {
                unsigned q = any ? row[0] + (unsigned)((b * 16 + lh * 8) * p.taps + tap) * (unsigned)p.M * 4u : CL_OUT;
                asm volatile("" : "+v"(q));
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    k.wf[u * 8 + e] = __builtin_amdgcn_raw_buffer_load_b32(rw, q, 0, 0);
                    q += w_step;
                }
            }
        }
        if (DATA) {
            // 8 lanes per row, four per unit; pieces that the last channel cuts, or that lie past it, start at the last four
            const int unit = c * 2 + ((lane & 7) >> 2), tap = cl_quot(unit, p.by_blocks), past = (unit - tap * blocks) * 16 + (lane & 3) * 4 + 4 - p.K;
            const unsigned at = (lane & 4 ? at_w[1] : at_w[0]) + (unsigned)((lane & 3) * 4 - (past > 0 ? past : 0)) * 4u;
#pragma unroll
            for (int q = 0; q < 4; q++) k.wd[q] = __builtin_amdgcn_raw_buffer_load_b128(rw, row[q] + at, 0, 0);
        }
    };
    floatx16 acc[1][1], sum;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[0][0][r] = sum[r] = 0.f;

    const int chunks = (p.units + 1) >> 1;
    int odd = 0;
    auto step = [&](Chunk& k, int c) {
        half8_t a[2], b[2];
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                b[u][e] = (_Float16)__builtin_bit_cast(float, k.xv[u * 8 + e]);
                if constexpr (!DATA && !IMAGE) a[u][e] = (_Float16)__builtin_bit_cast(float, k.wf[u * 8 + e]);
            }
        if constexpr (IMAGE) {
            a[0] = __builtin_bit_cast(half8_t, k.wd[0]);
            a[1] = __builtin_bit_cast(half8_t, k.wd[1]);
        }
        if constexpr (DATA) {
            const int unit = c * 2 + ((lane & 7) >> 2), tap = cl_quot(unit, p.by_blocks), at = (unit - tap * blocks) * 16 + (lane & 3) * 4, past = at + 4 - p.K;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                piece4 v = __builtin_bit_cast(piece4, k.wd[q]);
                if (p.K & 15) {
                    v = turn_back(v, past > 0 ? past : 0);
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = at + e < p.K ? v[e] : 0.f;
                }
                half4_t h;
#pragma unroll
                for (int e = 0; e < 4; e++) h[e] = (_Float16)v[e];
                *reinterpret_cast<half4_t*>(own + (q * 8 + (lane >> 3)) * SLICE_PITCH + (lane & 7) * 8) = h;
            }
        }
        if (c + NW < chunks) load(k, c + NW);
        if constexpr (DATA) {
            slice_wave_sync();
            const char* q = own + li * SLICE_PITCH + lh * 16;
            a[0] = *reinterpret_cast<const half8_t*>(q);
            a[1] = *reinterpret_cast<const half8_t*>(q + 32);
        }
        if (odd ^= 1) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                sum[r] += acc[0][0][r];
                acc[0][0][r] = 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < 2; u++) acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[u], b[u], acc[0][0], 0, 0, 0);
        if constexpr (DATA) slice_wave_sync();
    };
    Chunk k;
    if (wave < chunks) load(k, wave);
    for (int c = wave; c < chunks; c += NW) step(k, c);
#pragma unroll
    for (int r = 0; r < 16; r++) acc[0][0][r] += sum[r];

    const int active = chunks < NW ? chunks : NW;
    piece4* park = reinterpret_cast<piece4*>(lds);
    if (DATA) __syncthreads();
    if (wave < active) slice_park(park, acc, wave, lane);
    __syncthreads();
    if (wave >= 4 || px >= pixels) return;
    const int g = wave, m = m0 + g * 8 + lh * 4;
    piece4 v = slice_collect<1, 1, NW>(park, g, 0, active, lane);
    float* y = p.y + img * p.y_img + px;
    if (DATA) {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (__builtin_expect(v[e] != v[e] && m + e < p.M, 0)) {  // a zero in the place of a tap outside dy may have met an infinite weight
                bool edge = false;
                for (int tap = 0; tap < p.taps; tap++) {
                    const int r = cl_quot(tap, p.by_kw);
                    edge |= slice_tap<true>(p, h0, w0, r, tap - r * p.K_w) < 0;
                }
                if (edge) v[e] = slice_terms(p, xi, wi, h0, w0, m + e);
            }
    }
    float old[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int me = m + e < p.M ? m + e : p.M - 1;
        old[e] = DATA ? (p.accumulate ? y[(long)me * pixels] : 0.f) : p.bias ? p.bias[img * p.bias_sn + px * p.bias_sp + me * p.bias_sc] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float o = v[e] + old[e];
        if (p.relu) o = o > 0.f ? o : 0.f;
        if (m + e < p.M) y[(long)(m + e) * pixels] = o;
    }
}

// The image a forward's caller keeps, once per change of the weights: a thread per row and half a unit
__global__ __launch_bounds__(256) void conv_slices_image_kernel(_Float16* image, const float* __restrict__ w, int M, int K, int taps, int blocks, int rows, long halves) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;              // [copy][unit][half][row]
    if (i >= halves) return;
    const int m = (int)(i % rows), half = (int)(i / rows & 1);
    const long unit = i / rows / 2, copy = unit / (taps * blocks);
    const int u = (int)(unit - copy * taps * blocks), tap = u / blocks, c0 = (u - tap * blocks) * 16 + half * 8;
    half8_t h;
#pragma unroll
    for (int e = 0; e < 8; e++) h[e] = m < M && c0 + e < K ? (_Float16)w[((copy * K + c0 + e) * taps + tap) * M + m] : (_Float16)0.f;
    *reinterpret_cast<half8_t*>(image + (unit * rows + m) * 16 + half * 8) = h;
}

// ---- host side ----------------------------------------------------------------------------------------------------------
static ConvSliceArgs conv_slices_args(bool data, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w, size_t stride, size_t pad, size_t w_batch) {
    ConvSliceArgs a = {};
    const int Ho = (int)((H + 2 * pad - K_h) / stride + 1), Wo = (int)((W + 2 * pad - K_w) / stride + 1);
    a.M = (int)(data ? C : O); a.K = (int)(data ? O : C); a.taps = (int)(K_h * K_w); a.K_w = (int)K_w;
    a.Hx = data ? Ho : (int)H; a.Wx = data ? Wo : (int)W; a.Hr = data ? (int)H : Ho; a.Wr = data ? (int)W : Wo;
    a.stride = (int)stride; a.pad = (int)pad;
    const int blocks = (a.K + 15) / 16;
    a.units = a.taps * blocks;
    a.tiles_m = (a.M + 31) / 32;
    a.tiles = a.tiles_m * ((a.Hr * a.Wr + 31) / 32);
    a.total = a.tiles * (int)N;
    a.x_img = (long)a.K * a.Hx * a.Wx; a.y_img = (long)a.M * a.Hr * a.Wr; a.w_img = w_batch > 1 ? (long)C * a.taps * O : 0;
    a.x_bytes = (unsigned)(a.x_img * 4); a.w_bytes = (unsigned)(C * a.taps * O * 4);
    a.by_blocks = cl_div(blocks); a.by_kw = cl_div(a.K_w); a.by_tiles = cl_div(a.tiles); a.by_tiles_m = cl_div(a.tiles_m); a.by_wr = cl_div(a.Wr); a.by_stride = cl_div(a.stride);
    return a;
}

// Drawn on 350 layers of 1 to 32 images, 3 to 512 channels, 7 x 7 to 224 x 224 and kernels 1, 3, 5 and 7 (us a call, the ways before / here):
// - a wave's chain of chunks: up to 80 units, 130 where 100 tiles and more share the weights (1 x 336 x 16 x 16 -> 314 14.6 / 18.3, 189 units; 2 x 240 x 16 x 16
//   -> 66 12.1 / 11.4, 135)
// - what the tiles take in: 90 MB (16 x 64 x 12 x 48 -> 176, 255 MB, 13.1 / 17.6; 16 x 10 x 32 x 8 -> 224 5x5, 92 MB, 10.3 / 10.3), a data gradient 80
//   (10 x 16 x 48 x 48 <- 80, 133 MB, 15.6 / 10.7, but 4 x 104 x 64 x 64 <- 19, 151 MB, 10.7 / 13.7)
// - data gradients at strides, which multiply zeros here: up to 72 units (1 x 105 x 39 x 39 <- 126, 72, 9.7 / 9.2; 5x5 1 x 79 x 21 x 21 <- 40, 75, 9.6 / 9.8;
//   10 x 15 x 19 x 19 <- 194, 117, 11.5 / 13.3) and 60 MB, 45 MB where some CUs get two of the tiles (16 x 11 x 25 x 25 <- 48, 35 MB, 10.3 / 8.0;
//   4 x 26 x 46 x 46 <- 27 5x5, 268 tiles, 55 MB, 8.8 / 10.3), drawn on 45 more
// - tiles: 3300 and 1500 (16 x 11 x 80 x 80 -> 48 1x1, 6400, 20.5 / 17.3, but 8 x 5 x 80 x 80 -> 138, 8000, 24.2 / 24.8)
//   shared 1x1 forwards of more than 160 outputs 2000 (32 x 16 x 18 x 18 -> 192 8.6 / 10.7, 10 x 52 x 32 x 32 -> 320 9.9 / 11.1)
// - forwards of 1x1 at strides, which otherwise copy the pixels they look at first: 350 MB (10 x 400 x 150 x 150 -> 21 105 / 47, 4 x 288 x 158 x 158 -> 171 55 / 50)
//   not with a bias per pixel and more than 224 outputs where that and y are most of the traffic (8 x 20 x 80 x 80 -> 336 17.2 / 21.1, 4 x 14 x 112 x 112 -> 368
//   17.5 / 21.2; 16 x 17 x 66 x 66 -> 211 17.9 / 13.9)
// - 1x1 data gradients are one product already: only those of up to 8 channels, on which the streaming kernels are slow (16 x 8 x 88 x 88 <- 480 127 / 49)
static int conv_slices_shape(bool data, const ConvSliceArgs& a, bool one, size_t stride, bool pixel_bias) {
    const double mb = (double)a.total * a.units * 4096e-6;
    const int shape = a.total <= 512 && a.units > 8;                  // 8 waves where a CU gets one or two workgroups (8 x 240 x 8 x 8 -> 235 16.5 us with 4, 13.1 with 8)
    if (one && data && stride == 1) return a.M <= 8 && a.K >= 32 && mb <= 500 ? shape : -1;
    if (one && !data && stride > 1) return mb <= 350 && a.total <= 5000 && !(pixel_bias && a.units <= 2 && a.tiles_m >= 8 && a.total > 3300) ? shape : -1;
    if (one && !data && !a.w_img && a.tiles_m >= 6 && a.total > 2000) return -1;
    if (a.units > (a.total >= 100 ? 130 : 80)) return -1;
    if (data && stride > 1 && (a.units > 72 || mb > (a.total > 256 ? 45 : 60))) return -1;
    return mb <= (!data ? 90 : 80) && a.total <= (data ? 1500 : 3300) ? shape : -1;
}

// Estimated time in us of a forward that is no 1x1 at a stride, or a data gradient at stride 1, fitted on 1399 and 500 of them (11 % and 15 % off on average):
// a wave's chunks, what a second workgroup adds to them, and the lines that 32 pixels of a channel lie on, at a stride two to four.
static double conv_slices_cost(bool data, const ConvSliceArgs& a, int shape, bool pixel_bias) {
    const double r = (double)a.total / device_cu_count(), more = r > 1.0 ? r - 1.0 : 0.0, out = (double)a.y_img * (a.total / a.tiles) * 1e-6;
    const int nw = shape ? 8 : 4, two = shape && r > 1.0, lines = a.stride == 1 ? 0 : a.Wr >= 32 ? 1 : a.Wr >= 16 ? 2 : 3;
    const double chunks = (double)(((a.units + 1) / 2 + nw - 1) / nw);
    if (data) return shape ? 2.8 + chunks * (1.0 + 0.54 * two) + 0.0018 * a.total : 0.3 + 1.67 * chunks + r * (1.26 - 0.13 * chunks);
    const double first = shape ? 0.93 + 0.07 * lines : 0.54 + 0.19 * lines, next = shape ? two * (0.51 + 0.16 * lines) : 0.37 * more;
    return 2.7 + chunks * (first + next) + out * ((shape ? 1.8 : 0.9) + (pixel_bias ? 1.1 : 0.0));
}

int conv_slices_plan(ClDirection dir, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w, size_t stride, size_t pad, size_t w_batch, bool pixel_bias) {
    static const bool others = getenv("NZHIP_CONV_ROUTE") || getenv("NZHIP_CONV_DX") || getenv("NZHIP_CONV_1X1_GEMM") || getenv("NZHIP_CONV_TW") || getenv("NZHIP_CONV_BN");
    const char* env = getenv("NZHIP_CONV_SLICES");                    // read per call (tests, benchmarking): 0 never, 1 and 2 that shape wherever it fits
    // a run that asks for one of the other routes gets it
    if (!env && (others || getenv("NZHIP_CONV_CL") || getenv("NZHIP_CONV_WIDEN"))) return -1;
    // offsets of 32 bits inside an image and a weight copy; pieces of four along a data gradient's contraction
    const size_t lim = (size_t)1 << 28, Hp = H + 2 * pad, Wp = W + 2 * pad;
    if (!N || !H || !W || H >= 16384 || W >= 16384 || pad > 4096 || stride > 4096 || K_h > 4096 || K_w > 4096 || C >= lim || O >= lim || (dir == CL_DATA && O < 4) ||
        (C + 32) * H * W >= lim || (O + 32) * Hp * Wp >= lim || (C + 32) * Hp * Wp >= lim || (C + 32) * K_h * K_w * (O + 32) >= lim) return -1;
    const size_t Ho = (Hp - K_h) / stride + 1, Wo = (Wp - K_w) / stride + 1;
    if (N * ((C + O + 62) / 32 + 1) * ((H * W + Ho * Wo) / 32 + 2) >= lim) return -1;
    if (env) return atoi(env) >= 1 && atoi(env) <= 2 ? atoi(env) - 1 : -1;
    const bool data = dir == CL_DATA, one = K_h == 1 && K_w == 1;
    const ConvSliceArgs a = conv_slices_args(data, N, C, H, W, O, K_h, K_w, stride, pad, w_batch);
    const int shape = conv_slices_shape(data, a, one, stride, pixel_bias);
    if (shape < 0 || (one && (data || stride > 1)) || (data && stride > 1)) return shape;
    // Near those lines the copies are often ahead, most of all with few channels, whose units are filled up, and at strides: taken where this one's estimate is
    // 10 % below theirs, or just below with a weight copy per image, which they are slow on. Of 1399 forwards 121 were more than 5 % slower here than on the
    // ways before (16 x 112 x 16 x 16 -> 283 3x3 at stride 2 13.0 / 18.7, 2 x 3 x 107 x 107 -> 318 9.3 / 12.1, 32 x 7 x 11 x 11 -> 336 8.7 / 10.4), 32 are now, by 0.4 to 2 us;
    // of 347 gradients 18 (16 x 96 x 16 x 16 <- 4 7x7 8.6 / 10.8) and 4. Up to 64 outputs, 20 MB and 800 tiles this one is nearly always ahead.
    if ((data || a.tiles_m >= 3) && ((double)a.total * a.units * 4096e-6 > 20 || a.total > 800) && cl_conv_fits(dir, N, C, H, W, O, K_h, K_w, stride, pad, w_batch) &&
        conv_slices_cost(data, a, shape, pixel_bias) >= (!data && w_batch > 1 ? 1.0 : 0.9) * cl_conv_cost(dir, N, C, H, W, O, K_h, K_w, stride, pad, w_batch)) return -1;
    return shape;
}

int conv_slices_run(bool data, int shape, float* y, const float* x, const float* w, const float* bias, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w,
                    size_t stride, size_t pad, size_t w_batch, int64_t bias_sp, int64_t bias_sc, int64_t bias_sn, int relu, int accumulate, hipStream_t s) {
    ConvSliceArgs a = conv_slices_args(data, N, C, H, W, O, K_h, K_w, stride, pad, w_batch);
    a.y = y; a.x = x; a.w = w; a.bias = bias; a.bias_sp = bias_sp; a.bias_sc = bias_sc; a.bias_sn = bias_sn; a.relu = relu; a.accumulate = accumulate;
    ImageLease lease;
    int rc = NZHIP_OK;
    // (an image that its filled-up tiles and units make more than twice the size of the weights saves nothing)
    if (!data && image_kept_by_caller(PREPARED_CONV_W) && (size_t)a.units * a.tiles_m * 512 <= (size_t)a.w_bytes) {
        const int copies = w_batch > 1 ? (int)w_batch : 1, rows = a.tiles_m * 32;
        const uint64_t key[PREPARED_KEY_WORDS] = {0x51u | (uint64_t)K_h << 8 | (uint64_t)K_w << 24, reinterpret_cast<uintptr_t>(w), C, O, 0, 0, w_batch};
        rc = image_acquire(PREPARED_CONV_W, key, (size_t)copies * a.units * rows * 32, s, &lease);
        if (rc == NZHIP_E_NOMEM) {                                    // no memory to keep one: the weights as they lie
            lease = ImageLease();
            rc = NZHIP_OK;
        }
        if (rc) return rc;
        a.image = reinterpret_cast<const _Float16*>(lease.ptr);
        a.image_img = w_batch > 1 ? (long)a.units * rows * 16 : 0;
        if (lease.ptr && lease.fill) {
            const long halves = (long)copies * a.units * rows * 2;
            hipLaunchKernelGGL(conv_slices_image_kernel, dim3((unsigned)((halves + 255) / 256)), dim3(256), 0, s, reinterpret_cast<_Float16*>(lease.ptr), w, a.M, a.K, a.taps,
                               (a.K + 15) / 16, rows, halves);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) rc = set_hip_error(e, "conv slices image kernel launch");
        }
    }
    const bool filled = rc == NZHIP_OK;
    if (rc == NZHIP_OK) {
        const int nw = shape ? 8 : 4;
        auto kfn = data      ? (shape ? conv_slices_kernel<true, false, 8> : conv_slices_kernel<true, false, 4>)
                   : a.image ? (shape ? conv_slices_kernel<false, true, 8> : conv_slices_kernel<false, true, 4>)
                             : (shape ? conv_slices_kernel<false, false, 8> : conv_slices_kernel<false, false, 4>);
        hipLaunchKernelGGL(kfn, dim3((unsigned)a.total), dim3(nw * 64), (size_t)nw * 4096, s, a);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) rc = set_hip_error(e, "conv slices kernel launch");
    }
    const int rc2 = lease.ptr ? image_release(lease, s, filled) : NZHIP_OK;
    return rc ? rc : rc2;
}

}  // namespace nzhip
