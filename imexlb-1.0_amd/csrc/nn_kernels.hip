// nn_kernels.hip -- gfx950 kernels of the warm-start network: a small
// convolutional encoder-decoder trained and run on the GPU by these kernels
// (C ABI in include/imexlb_nn.h).  Tensors are FP32, NCHW, in device memory
// the caller owns; every launch goes to the given stream.
//
// conv3x3 (padding 1, stride 1) in FP32 runs on the matrix cores (k_conv3
// below); the data gradient is the same kernel on the flipped, transposed
// weights; the weight gradient (k_conv3_dw) sums a 16x16 tile of pixels over
// the batch on the matrix cores, and the tiles' sums are added in order or
// with atomics.
//
// Inference in BF16 (k_conv3_bf16): activations NHWC bf16, weights packed
// [CI/8][tap][CO][8 ci] bf16, products on the matrix cores
// (v_mfma_f32_32x32x16_bf16, FP32 accumulation), bias, ReLU and the
// rounding to bf16 (round to nearest even) fused into the store, with the
// pooled copy; a decoder layer reads the upsampled and the skip channels from
// their own buffers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <initializer_list>
#include <mutex>
#include <string>
#include <type_traits>

#include "../../include/imexlb_nn.h"
#include "context.hpp"

namespace imexlb_nn {

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// Order of the blocks of a 1D grid: blocks are dealt to the 8 XCDs in turn,
// so this gives each XCD one contiguous run of tiles (blocks that share
// input or weights share an L2).
__device__ __forceinline__ uint32_t xcd_run(uint32_t b, uint32_t nb)
{
    const uint32_t per = nb / 8u;
    return b < per * 8u ? (b % 8u) * per + b / 8u : b;
}

// 3x3 convolution, padding 1, as a matrix product over k = 9 ci + tap with
// v_mfma_f32_32x32x2_f32.  That instruction adds its two products to the
// accumulator one after the other, each as an FMA (compared bit for bit with
// a chain of FMAs, subnormals included), so taking k in order gives exactly
// the sum of a loop over input channels and taps.
//
// Bound by the matrix cores (157 TFLOP/s; a plain FMA loop has half).  A
// block computes 4 MT (32 / TC) rows x TC columns of pixels for 32 NT output
// channels, a wave MT groups of 32 pixels; rows of the product are output
// channels and columns pixels, so a half-wave stores 32 consecutive pixels.
// Eight input channels at a time (the tile with its halo, and the weights
// [k][co]) go through two LDS buffers in turn, fetched into registers while
// the previous eight are multiplied; every operand is one 32-bit LDS read
// without bank conflicts, read one product ahead.  The loads take no branch:
// one per load made each wait for the one before (80 against 115 TFLOP/s).
// Against one thread per pixel with 16 accumulators and FMAs: 96 -> 32
// channels, 8 x 128 x 512: 603 to 248 us (117 TFLOP/s); 64 -> 64, 8 x 64 x
// 256: 221 to 93 us; 256 -> 256, 8 x 16 x 64: 475 to 99 us; 256 -> 256, 1 x
// 16 x 64: 429 to 59 us.
constexpr int CIB = 8;  // input channels per LDS chunk

//
// The output goes to channels of a buffer with ototal of them per image
// (out points at the first).  DGRAD: w is [CI][CO][3][3], read flipped and
// transposed -- the data gradient of a layer from CO to CI channels -- and,
// with a gate (gtotal channels per image), the value is kept only where the
// gate is positive: the ReLU of the layer before.
// FEW: at most 6 input channels, whose missing pairs are left out (8 x 512 x
// 512: 1 -> 1 channels 100 to 58 us, 4 -> 1 99 to 73; the test costs the others
// 3 %, the products being scheduled pair by pair).
template <int MT, int NT, int TC, bool DGRAD, bool FEW>
__global__ __launch_bounds__(256) void k_conv3(const float *__restrict__ in, const float *__restrict__ w,
                                               const float *__restrict__ bias, float *__restrict__ out, int ototal,
                                               const float *__restrict__ gate, int gtotal, int CI, int CO, int H, int W,
                                               int relu, uint32_t ntx, uint32_t nty, uint32_t ncob)
{
    constexpr int GR = 32 / TC;  // rows of a 32-pixel group
    constexpr int TR = 4 * MT * GR, IR = TR + 2, IC = TC + 2, BN = 32 * NT, WS = BN + 1;
    constexpr int NP = (IR * IC + 63) / 64, NW = (BN + 2) / 3;
    __shared__ float s_in[2][CIB * IR * IC];
    __shared__ float s_w[2][CIB * 9 * WS];
    __shared__ float s_b[BN];
    const int tid = int(threadIdx.x), lane = tid % 64, wave = tid / 64;
    const int m = lane % 32, hk = lane / 32;  // operand row / column and which of the two k
    uint32_t blk = xcd_run(blockIdx.x, gridDim.x);
    const int co0 = int(blk % ncob) * BN;
    blk /= ncob;
    const int x0 = int(blk % ntx) * TC;
    blk /= ntx;
    const int y0 = int(blk % nty) * TR;
    const int64_t n = blk / nty, HW = int64_t(H) * W;
    const float *const img = in + n * CI * HW;

    // Staging.  A wave brings two channels of the tile with its halo; a
    // lane's pixels are the same for every channel.  Weights lie k = 9 ci +
    // tap fastest: a thread brings one k of every third output channel.
    // Loads have no branches: lanes with nothing to load read a valid
    // neighbour and drop it.
    int64_t ioff[NP];
    bool iok[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int p = lane + 64 * i, yy = y0 + p / IC - 1, xx = x0 + p % IC - 1;
        iok[i] = p < IR * IC && yy >= 0 && yy < H && xx >= 0 && xx < W;
        ioff[i] = iok[i] ? int64_t(yy) * W + xx : int64_t(y0) * W + x0;
    }
    const int ch = __builtin_amdgcn_readfirstlane(wave * 2);
    const int wk = tid % 72, wc = tid / 72;  // threads from 216 on repeat others' loads
    const int wlast = (min(co0 + BN, CO) - 1 - co0 - min(wc, CO - 1 - co0)) / 3;
    const int wco = co0 + min(wc, CO - 1 - co0);
    const float *const wrow = DGRAD ? w + int64_t(wco) * 9 + 8 - wk % 9 : w + int64_t(wco) * CI * 9;
    float xin[2][NP], xw[NW];
    auto load = [&](int c0) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const float *const pl = img + int64_t(min(c0 + ch + c, CI - 1)) * HW;
#pragma unroll
            for (int i = 0; i < NP; ++i) xin[c][i] = pl[ioff[i]];
        }
        const float *const p = wrow + (DGRAD ? min(c0 + wk / 9, CI - 1) * int64_t(CO) * 9
                                             : min(int64_t(c0) * 9 + wk, int64_t(CI) * 9 - 1));
#pragma unroll
        for (int i = 0; i < NW; ++i) xw[i] = p[min(i, wlast) * (DGRAD ? 27 : int64_t(27) * CI)];
    };
    auto store = [&](int buf, int c0) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const bool live = c0 + ch + c < CI;
#pragma unroll
            for (int i = 0; i < NP; ++i)
                if (lane + 64 * i < IR * IC)
                    s_in[buf][(ch + c) * (IR * IC) + lane + 64 * i] = live && iok[i] ? xin[c][i] : 0.0f;
        }
        if (tid < 216) {
            const bool live = wk < (CI - c0) * 9;
#pragma unroll
            for (int i = 0; i < NW; ++i)
                if (wc + 3 * i < BN) s_w[buf][wk * WS + wc + 3 * i] = live ? xw[i] : 0.0f;
        }
    };
    // where the lane's pixel operand of product i of a channel pair lies:
    // its k is 2 i + hk, i.e. channel k / 9 of the pair and tap k % 9
    int bo[9];
    const int px = (wave * MT * GR + m / TC) * IC + m % TC;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const int k0 = 2 * i, k1 = 2 * i + 1;
        const int o0 = k0 / 9 * (IR * IC) + k0 % 9 / 3 * IC + k0 % 3;
        const int o1 = k1 / 9 * (IR * IC) + k1 % 9 / 3 * IC + k1 % 3;
        bo[i] = px + (hk ? o1 : o0);
    }
    const int ao = hk * WS + m;
    f32x16 acc[NT][MT] = {};
    if (tid < BN) s_b[tid] = bias && co0 + tid < CO ? bias[co0 + tid] : 0.0f;

    load(0);
    store(0, 0);
    __syncthreads();
    int buf = 0;
    for (int c0 = 0; c0 < CI; c0 += CIB) {
        const bool more = c0 + CIB < CI;
        if (more) load(c0 + CIB);
        const float *const si = s_in[buf], *const sw = s_w[buf];
        // operands of product k2 of the chunk (k = 2 k2 + hk), read one
        // product ahead of their use
        float a[2][NT], b[2][MT];
        auto fetch = [&](int k2, float(&fa)[NT], float(&fb)[MT]) {
#pragma unroll
            for (int t = 0; t < NT; ++t) fa[t] = sw[ao + 2 * k2 * WS + 32 * t];
#pragma unroll
            for (int t = 0; t < MT; ++t) fb[t] = si[bo[k2 % 9] + k2 / 9 * 2 * (IR * IC) + t * GR * IC];
        };
        fetch(0, a[0], b[0]);
#pragma unroll
        for (int k2 = 0; k2 < CIB * 9 / 2; ++k2) {
            if (FEW && k2 % 9 == 0 && k2 * 2 >= CI * 9) break;  // (pairs of channels past the last)
            if (k2 + 1 < CIB * 9 / 2) fetch(k2 + 1, a[(k2 + 1) % 2], b[(k2 + 1) % 2]);
#pragma unroll
            for (int s = 0; s < NT; ++s)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    acc[s][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[k2 % 2][s], b[k2 % 2][t], acc[s][t], 0, 0, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, NT + MT, 0);  // the reads of the next product,
            __builtin_amdgcn_sched_group_barrier(0x008, NT * MT, 0);  // then the products of this one
        }
        if (more) store(buf ^ 1, c0 + CIB);  // its last readers passed the barrier before this chunk
        __syncthreads();
        buf ^= 1;
    }
    // lane holds D[channel 8 (j/4) + 4 hk + j%4][pixel m] of each 32x32 tile
    const int x = x0 + m % TC;
    if (x >= W) return;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int y = y0 + (wave * MT + t) * GR + m / TC;
        if (y >= H) continue;
        float *const o = out + (n * ototal + co0) * HW + int64_t(y) * W + x;
        const float *const g = DGRAD && gate ? gate + (n * gtotal + co0) * HW + int64_t(y) * W + x : nullptr;
#pragma unroll
        for (int s = 0; s < NT; ++s) {
            float gv[16];  // all gate values in flight before the first is used
            if (DGRAD && g) {
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    gv[j] = g[min(32 * s + 8 * (j / 4) + 4 * hk + j % 4, CO - 1 - co0) * HW];
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int co = 32 * s + 8 * (j / 4) + 4 * hk + j % 4;
                float v = acc[s][t][j] + s_b[co];
                if (relu) v = v > 0.0f ? v : 0.0f;
                if (DGRAD && g) v = gv[j] > 0.0f ? v : 0.0f;
                if (co0 + co < CO) o[co * HW] = v;
            }
        }
    }
}

// wt[ci][co][8-k] = w[co][ci][k]: the data gradient as a forward conv
__global__ void k_flip(const float *__restrict__ w, float *__restrict__ wt, int CI, int CO)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= int64_t(CO) * CI * 9) return;
    const int k = int(i % 9), ci = int((i / 9) % CI), co = int(i / (9 * int64_t(CI)));
    wt[(int64_t(ci) * CO + co) * 9 + (8 - k)] = w[i];
}

// db[c] = sum of dout over batch and pixels (one block per channel): thread
// t adds pixels t, t + 256, ... of image after image, then a tree over the
// threads.  Bound by the latency of its loads (one channel's values pass
// through one CU): kBias of them are in flight per thread, the additions
// keep their order.  32 channels, 8 x 128 x 512: 505 us with one load in
// flight, 76 us now.
constexpr int kBias = 64;
__device__ __forceinline__ void bias_sum(const float *__restrict__ dout, float *__restrict__ db, int N, int C,
                                         int64_t HW, int c, float *red)
{
    const int64_t rows = (HW + 255) / 256;  // of 256 pixels per image, the last one ragged
    const float *p = dout + c * HW + threadIdx.x;
    const int64_t next = C * HW - rows * 256;  // from past the last row to the next image's first
    int64_t left = N * rows, i = 0;
    const bool tail = (rows - 1) * 256 + threadIdx.x < HW;  // this thread's pixel of the last row exists
    float s = 0.0f;
    const auto sum = [&](auto count) {
        constexpr int K = decltype(count)::value;
        for (; left >= K; left -= K) {
            float v[K];
            bool ok[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const bool last = i + 1 == rows;
                ok[k] = !last || tail;
                v[k] = p[ok[k] ? 0 : -int64_t(threadIdx.x)];  // (no branch: a missing pixel reads its row's first)
                p += last ? next + 256 : 256;
                i = last ? 0 : i + 1;
            }
#pragma unroll
            for (int k = 0; k < K; ++k) s += ok[k] ? v[k] : 0.0f;
        }
    };
    sum(std::integral_constant<int, kBias>{});
    sum(std::integral_constant<int, 8>{});
    sum(std::integral_constant<int, 1>{});
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (int(threadIdx.x) < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) db[c] = red[0];
    __syncthreads();  // (red is used again)
}

__global__ __launch_bounds__(256) void k_bias_grad(const float *__restrict__ dout, float *__restrict__ db, int N,
                                                   int C, int64_t HW)
{
    __shared__ float red[256];
    bias_sum(dout, db, N, C, HW, int(blockIdx.x), red);
}

constexpr int TS = 16;  // pixel tile edge of the weight gradient
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Weight gradient of one 16x16 tile of pixels, summed over the batch: for
// each tap a matrix product over the pixels (image after image, row after
// row) of the output gradient's channels and the shifted input's, with
// v_mfma_f32_16x16x4_f32, which adds its four products in order as FMAs --
// exactly the sum of a loop over the pixels.
// partial == nullptr: add to dw with atomics; otherwise write the block's
// sums to partial[blockIdx.x][co][ci][9] for k_dw_reduce (fixed order).
//
// Bound by the matrix cores (157 TFLOP/s).  A block takes 16 GCO output x 16
// GCI input channels, a wave 16 x 16 of them and all 9 taps; with fewer than
// four such groups the waves share the taps.  Half a tile (8 rows) of an
// image goes through LDS at a time, fetched into registers while the
// previous half is multiplied; 32 x 32 channels take 50 KB, three blocks on a
// CU.  Against one (co, ci) pair per thread and FMAs: 32 -> 32 channels, 8 x
// 128 x 512: 351 to 121 us; 96 -> 32: 917 to 281 us (103 TFLOP/s); 256 ->
// 256, 8 x 16 x 64: 274 to 112 us; 4 -> 32, 8 x 128 x 512: 247 to 67 us.
template <int GCO, int GCI>
__global__ __launch_bounds__(256) void k_conv3_dw(const float *__restrict__ in, const float *__restrict__ dout,
                                                  float *__restrict__ dw, int N, int CI, int CO, int H, int W,
                                                  float *__restrict__ partial, float *__restrict__ db)
{
    constexpr int NTAP = GCO * GCI == 4 ? 9 : GCO * GCI == 2 ? 5 : 3;  // taps per wave
    constexpr int HR = TS / 2, IC = TS + 2, IP = (HR + 2) * IC, GP = HR * TS;
    // channel strides of 2 (mod 32): the 16 channels x 2 pixels of a
    // half-wave read fall in 32 banks
    constexpr int SI = 226, SG = 162;
    __shared__ float s_in[GCI * 16 * SI];
    __shared__ float s_g[GCO * 16 * SG];
    const int tid = int(threadIdx.x), lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int m = lane % 16, kk = lane / 16;  // operand row / column, pixel of four
    // with db, the first row of blocks sums the bias gradient (the waits of
    // those few chains of additions pass while the others multiply)
    if (db && blockIdx.y == 0) {
        for (int c = int(blockIdx.x); c < CO; c += int(gridDim.x)) bias_sum(dout, db, N, CO, int64_t(H) * W, c, s_in);
        return;
    }
    const int by = int(blockIdx.y) - (db ? 1 : 0);
    const int ntx = (W + TS - 1) / TS;
    const int x0 = int(blockIdx.x) % ntx * TS, y0 = int(blockIdx.x) / ntx * TS;
    const int nci = (CI + 16 * GCI - 1) / (16 * GCI);
    const int co0 = by / nci * (16 * GCO), ci0 = by % nci * (16 * GCI);
    const int wco = wave % GCO, wci = wave / GCO % GCI, tap0 = wave / (GCO * GCI) * NTAP;
    const int64_t HW = int64_t(H) * W;

    // Staging: half a tile (8 rows) of one image; a wave brings every fourth
    // channel.  Channels past the end repeat the last one (their sums are
    // not stored); pixels outside the image are zero.
    constexpr int NI = (IP + 63) / 64, NG = GP / 64;
    float xi[GCI * 4][NI], xg[GCO * 4][NG];
    bool iok[NI], gok[NG];
    auto load = [&](int n, int h) {
        int64_t io[NI], go[NG];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int p = lane + 64 * i, yy = y0 + h * HR + p / IC - 1, xx = x0 + p % IC - 1;
            iok[i] = p < IP && yy >= 0 && yy < H && xx >= 0 && xx < W;
            io[i] = iok[i] ? int64_t(yy) * W + xx : 0;
        }
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const int p = lane + 64 * i, yy = y0 + h * HR + p / TS, xx = x0 + p % TS;
            gok[i] = yy < H && xx < W;
            go[i] = gok[i] ? int64_t(yy) * W + xx : 0;
        }
#pragma unroll
        for (int c = 0; c < GCI * 4; ++c) {
            const float *const pl = in + (int64_t(n) * CI + min(ci0 + wave + 4 * c, CI - 1)) * HW;
#pragma unroll
            for (int i = 0; i < NI; ++i) xi[c][i] = pl[io[i]];
        }
#pragma unroll
        for (int c = 0; c < GCO * 4; ++c) {
            const float *const pl = dout + (int64_t(n) * CO + min(co0 + wave + 4 * c, CO - 1)) * HW;
#pragma unroll
            for (int i = 0; i < NG; ++i) xg[c][i] = pl[go[i]];
        }
    };
    f32x4 acc[NTAP] = {};
    int bo[NTAP];  // the tap's offset in the lane's input channel
#pragma unroll
    for (int t = 0; t < NTAP; ++t) {
        const int tap = min(tap0 + t, 8);  // (a wave with fewer taps repeats the last, not stored)
        bo[t] = (wci * 16 + m) * SI + tap / 3 * IC + tap % 3 + kk;
    }
    const int ao = (wco * 16 + m) * SG + kk;
    const int halves = y0 + HR < H ? 2 : 1;

    load(0, 0);
    for (int n = 0, h = 0; n < N;) {
        __syncthreads();  // the previous part has been multiplied
#pragma unroll
        for (int c = 0; c < GCI * 4; ++c)
#pragma unroll
            for (int i = 0; i < NI; ++i)
                if (lane + 64 * i < IP) s_in[(wave + 4 * c) * SI + lane + 64 * i] = iok[i] ? xi[c][i] : 0.0f;
#pragma unroll
        for (int c = 0; c < GCO * 4; ++c)
#pragma unroll
            for (int i = 0; i < NG; ++i) s_g[(wave + 4 * c) * SG + lane + 64 * i] = gok[i] ? xg[c][i] : 0.0f;
        __syncthreads();
        const int rows = min(HR, H - y0 - h * HR);
        if (++h == halves) {
            h = 0;
            ++n;
        }
        if (n < N) load(n, h);
        // 4 pixels per product, in pixel order; operands read one product
        // ahead (past the last row: read, not used)
        float a[2], b[2][NTAP];
        a[0] = s_g[ao];
#pragma unroll
        for (int t = 0; t < NTAP; ++t) b[0][t] = s_in[bo[t]];
        for (int r = 0; r < rows; ++r) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int nx = (g + 1) % 2, ro = g == 3 ? r + 1 : r, go = (g + 1) % 4 * 4;
                a[nx] = s_g[ao + ro * TS + go];
#pragma unroll
                for (int t = 0; t < NTAP; ++t) b[nx][t] = s_in[bo[t] + ro * IC + go];
#pragma unroll
                for (int t = 0; t < NTAP; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[g % 2], b[g % 2][t], acc[t], 0, 0, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
                for (int t = 0; t < NTAP; ++t) {  // one read between two products
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                }
            }
        }
    }
    // lane holds D[co 4 kk + j][ci m]
    const int ci = ci0 + wci * 16 + m;
    if (ci >= CI) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int co = co0 + wco * 16 + 4 * kk + j;
        if (co >= CO) continue;
        const int64_t o = (int64_t(co) * CI + ci) * 9;
        float *const pb = partial ? partial + int64_t(blockIdx.x) * CO * CI * 9 + o : dw + o;
#pragma unroll
        for (int t = 0; t < NTAP; ++t) {
            if (tap0 + t >= 9) continue;
            if (partial)
                pb[tap0 + t] = acc[t][j];
            else
                atomicAdd(&pb[tap0 + t], acc[t][j]);
        }
    }
}

// dw[i] += sum over tiles b = 0..nb-1 of partial[b][i], in that order, kRed
// loads in flight per thread
constexpr int kRed = 32;
__global__ __launch_bounds__(64) void k_dw_reduce(const float *__restrict__ partial, float *__restrict__ dw, int64_t nb,
                                                  int64_t n)
{
    const int64_t i = int64_t(blockIdx.x) * 64 + threadIdx.x;
    if (i >= n) return;
    float s = 0.0f;
    int64_t b = 0;
    for (; b + kRed <= nb; b += kRed) {
        float v[kRed];
#pragma unroll
        for (int k = 0; k < kRed; ++k) v[k] = partial[(b + k) * n + i];
#pragma unroll
        for (int k = 0; k < kRed; ++k) s += v[k];
    }
    for (; b < nb; ++b) s += partial[b * n + i];
    dw[i] += s;
}

__global__ void k_relu_bwd(const float *__restrict__ out, const float *__restrict__ dout, float *__restrict__ dz,
                           int64_t n)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) dz[i] = out[i] > 0.0f ? dout[i] : 0.0f;
}

// K consecutive values, as one access where the buffers allow it (A)
template <int K>
struct Px {
    float v[K];
};
template <bool A, int K>
__device__ __forceinline__ Px<K> ld_px(const float *p)
{
    if constexpr (A && K == 4)
        return __builtin_bit_cast(Px<K>, *reinterpret_cast<const float4 *>(p));
    else if constexpr (A && K == 2)
        return __builtin_bit_cast(Px<K>, *reinterpret_cast<const float2 *>(p));
    Px<K> r;
#pragma unroll
    for (int k = 0; k < K; ++k) r.v[k] = p[k];
    return r;
}
template <bool A, int K>
__device__ __forceinline__ void st_px(float *p, const Px<K> &v)
{
    if constexpr (A && K == 4)
        *reinterpret_cast<float4 *>(p) = __builtin_bit_cast(float4, v);
    else if constexpr (A && K == 2)
        *reinterpret_cast<float2 *>(p) = __builtin_bit_cast(float2, v);
    else {
#pragma unroll
        for (int k = 0; k < K; ++k) p[k] = v.v[k];
    }
}

// Pooling and upsampling: a thread takes one low-resolution pixel of one
// channel of one image, or two with 8- and 16-byte accesses (A) where w is even
// and the buffers are aligned; their place by three 32-bit multiplications
// (64-bit divisions cost more than the memory access).  Bound by HBM: the three
// upsamplings of a training step of 8 cases on 128 x 512 take 45 us in all; 8 x
// 64 channels of 64 x 256, gradients with the ReLU 29 us, joined with the skip
// connection 76.  A wave per row, its place by scalar divisions, was as fast
// from 128 columns on (78 us for the join, 64 columns 18 against 8) and idle on
// narrow ones (40 x 256 of 64 x 4: 165 us against 11); it takes the calls whose
// values 32 bits do not count.
struct LowRes {
    int N, C, h, w;
    uint32_t items;  // threads with work; 0 where they are 2^31 or more
    FastDiv per_row, rows, chans;
};
template <bool A, class F>
__device__ __forceinline__ void for_values(const LowRes &g, F f)
{
    constexpr int V = A ? 2 : 1;
    const auto div = [](uint32_t n, const FastDiv &d) { return (__umulhi(n, d.m) + n) >> d.s; };  // n < 2^31
    if (g.items) {
        const uint32_t i = blockIdx.x * 256u + threadIdx.x;
        if (i >= g.items) return;
        const uint32_t r = div(i, g.per_row), nc = div(r, g.rows), n = div(nc, g.chans);
        f(int64_t(n), int(nc - n * uint32_t(g.C)), int(r - nc * uint32_t(g.h)), int(i - r * uint32_t(g.w / V)) * V);
        return;
    }
    const int64_t rows = int64_t(g.N) * g.C * g.h;
    for (int64_t r = int64_t(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / 64); r < rows;
         r += int64_t(gridDim.x) * 4) {
        const int64_t nc = r / g.h, n = nc / g.C;
        const int y = int(r - nc * g.h), c = int(nc - n * g.C);
        for (int x = int(threadIdx.x % 64) * V; x < g.w; x += 64 * V) f(n, c, y, x);
    }
}

// 2x2 average pool of channels [coff, coff + C) of in [N][Ctot][2h][2w]
// (in points at channel coff) into out [N][C][h][w]
template <bool A>
__global__ __launch_bounds__(256) void k_pool2(const float *__restrict__ in, int Ctot, float *__restrict__ out, LowRes lr)
{
    constexpr int V = A ? 2 : 1;
    const int C = lr.C, h = lr.h, w = lr.w;
    for_values<A>(lr, [&](int64_t n, int c, int y, int x) {
        const float *p = in + ((n * Ctot + c) * 2 * h + 2 * y) * (2 * int64_t(w)) + 2 * x;
        const Px<2 * V> a = ld_px<A, 2 * V>(p), b = ld_px<A, 2 * V>(p + 2 * int64_t(w));
        Px<V> o;
#pragma unroll
        for (int k = 0; k < V; ++k) o.v[k] = 0.25f * ((a.v[2 * k] + a.v[2 * k + 1]) + (b.v[2 * k] + b.v[2 * k + 1]));
        st_px<A, V>(out + ((n * C + c) * h + y) * int64_t(w) + x, o);
    });
}

// Gradient of the pool, din [N][C][2h][2w]: 0.25 dout of the pixel's cell,
// plus skip (stot channels per image) if given, where gate (gtot channels
// per image) is positive if given.
template <bool A>
__global__ __launch_bounds__(256) void k_pool2_bwd(const float *__restrict__ dout, const float *__restrict__ skip,
                                                   int stot, const float *__restrict__ gate, int gtot,
                                                   float *__restrict__ din, LowRes lr)
{
    constexpr int V = A ? 2 : 1;
    const int C = lr.C, h = lr.h, w = lr.w;
    const int64_t W = 2 * int64_t(w);
    for_values<A>(lr, [&](int64_t n, int c, int y, int x) {
        const Px<V> g = ld_px<A, V>(dout + ((n * C + c) * h + y) * int64_t(w) + x);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int64_t row = 2 * y + k;
            Px<2 * V> o, s, a;
            if (skip) s = ld_px<A, 2 * V>(skip + ((n * stot + c) * 2 * h + row) * W + 2 * x);
            if (gate) a = ld_px<A, 2 * V>(gate + ((n * gtot + c) * 2 * h + row) * W + 2 * x);
#pragma unroll
            for (int j = 0; j < 2 * V; ++j) {
                o.v[j] = 0.25f * g.v[j / 2];
                if (skip) o.v[j] = o.v[j] + s.v[j];
                if (gate && !(a.v[j] > 0.0f)) o.v[j] = 0.0f;
            }
            st_px<A, 2 * V>(din + ((n * C + c) * 2 * h + row) * W + 2 * x, o);
        }
    });
}

// nearest 2x upsample: in [N][C][h][w] -> C channels of out [N][Ctot][2h][2w]
// (out points at the first)
template <bool A>
__global__ __launch_bounds__(256) void k_up2(const float *__restrict__ in, float *__restrict__ out, int Ctot, LowRes lr)
{
    constexpr int V = A ? 2 : 1;
    const int C = lr.C, h = lr.h, w = lr.w;
    const int64_t W = 2 * int64_t(w);
    for_values<A>(lr, [&](int64_t n, int c, int y, int x) {
        const Px<V> v = ld_px<A, V>(in + ((n * C + c) * h + y) * int64_t(w) + x);
        Px<2 * V> o;
#pragma unroll
        for (int j = 0; j < 2 * V; ++j) o.v[j] = v.v[j / 2];
        float *const p = out + ((n * Ctot + c) * 2 * h + 2 * y) * W + 2 * x;
        st_px<A, 2 * V>(p, o);
        st_px<A, 2 * V>(p + W, o);
    });
}

// its gradient, where gate (gtot channels per image) is positive if given
template <bool A>
__global__ __launch_bounds__(256) void k_up2_bwd(const float *__restrict__ dout, int Ctot,
                                                 const float *__restrict__ gate, int gtot, float *__restrict__ din,
                                                 LowRes lr)
{
    constexpr int V = A ? 2 : 1;
    const int C = lr.C, h = lr.h, w = lr.w;
    for_values<A>(lr, [&](int64_t n, int c, int y, int x) {
        const float *p = dout + ((n * Ctot + c) * 2 * h + 2 * y) * (2 * int64_t(w)) + 2 * x;
        const Px<2 * V> a = ld_px<A, 2 * V>(p), b = ld_px<A, 2 * V>(p + 2 * int64_t(w));
        Px<V> o, t;
        if (gate) t = ld_px<A, V>(gate + ((n * gtot + c) * h + y) * int64_t(w) + x);
#pragma unroll
        for (int k = 0; k < V; ++k) {
            o.v[k] = (a.v[2 * k] + a.v[2 * k + 1]) + (b.v[2 * k] + b.v[2 * k + 1]);
            if (gate && !(t.v[k] > 0.0f)) o.v[k] = 0.0f;
        }
        st_px<A, V>(din + ((n * C + c) * h + y) * int64_t(w) + x, o);
    });
}

// dst[:, dcoff+c] (=|+=) src[:, scoff+c] for c < C
__global__ void k_copy_ch(const float *__restrict__ src, int sctot, int scoff, float *__restrict__ dst, int dctot,
                          int dcoff, int N, int C, int64_t HW, int accumulate)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= int64_t(N) * C * HW) return;
    const int64_t p = i % HW;
    const int c = int((i / HW) % C), n = int(i / (HW * C));
    const float v = src[(int64_t(n) * sctot + scoff + c) * HW + p];
    float *d = dst + (int64_t(n) * dctot + dcoff + c) * HW + p;
    *d = accumulate ? *d + v : v;
}

// grad = 2 (pred - target) / n;  loss += sum (pred - target)^2 / n.  At most
// kMseBlocks blocks stride over the values and add their sum (kept in FP64)
// to the loss with one atomic each: with a block per 256 values the atomics
// on one word took most of the time and rounded the loss thousands of times
// (1.57 M values: 81 us and up to 3e-6 off; now 10 us and under 1e-7).
constexpr int64_t kMseBlocks = 128;
__global__ __launch_bounds__(1024) void k_mse(const float *__restrict__ pred, const float *__restrict__ target,
                                              float *__restrict__ grad, int64_t n, float *__restrict__ loss)
{
    __shared__ double red[16];
    double s = 0.0;
#pragma unroll 4
    for (int64_t i = int64_t(blockIdx.x) * 1024 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 1024) {
        const float d = pred[i] - target[i];
        if (grad) grad[i] = 2.0f * d / float(n);
        s += double(d * d / float(n));
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = s;
    __syncthreads();
    if (threadIdx.x == 0 && loss) {
        for (int k = 1; k < 16; ++k) s += red[k];
        atomicAdd(loss, float(s));
    }
}

__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m, float *__restrict__ v,
                       int64_t n, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (__builtin_sqrtf(vi / c2) + eps);
}

// ------------------------------------------------------------ BF16 inference
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// FP32 -> bf16, round to nearest even (NaN kept quiet)
__device__ __forceinline__ uint16_t to_bf16(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return uint16_t((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return uint16_t(u >> 16);
}

// two values to bf16 in one instruction, the same rounding (NaN quiet)
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

__device__ __forceinline__ float from_bf16(uint32_t h) { return __uint_as_float(h << 16); }

// average of four pixels' 8 channels, in FP32, rounded to bf16
__device__ __forceinline__ uint4 average4(uint4 a, uint4 b, uint4 c, uint4 d)
{
    const uint4 v[4] = {a, b, c, d};
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float avg[2];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            float s[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t word = k == 0 ? v[q].x : k == 1 ? v[q].y : k == 2 ? v[q].z : v[q].w;
                s[q] = from_bf16(half ? word >> 16 : word & 0xffffu);
            }
            avg[half] = 0.25f * ((s[0] + s[1]) + (s[2] + s[3]));
        }
        o[k] = pack2(avg[0], avg[1]);
    }
    return make_uint4(o[0], o[1], o[2], o[3]);
}

// slot of 8-channel group g of the pixel in column c, in the pixel's run of G
// slots in LDS: turned by the column so that 8 neighbours' slots of one group
// fall in different banks
template <int G>
__device__ __forceinline__ int turn(int g, int c)
{
    return G == 4 ? g ^ ((c >> 1) & 3) : g ^ ((c >> 2) & 1);
}

// The store of a tile of MT groups of 32 pixels and 32 channels per wave, WY
// waves down and 4 / WY across the channels: bias, ReLU, and for bf16 output
// through LDS (every wave's reads of it are over) so that the stores are 16
// bytes wide, with the pooled copy if asked for.
template <int MT, int WY, int TC>
__device__ __forceinline__ void conv_store(const f32x16 (&acc)[MT], uint4 *sh, const float *__restrict__ bias,
                                           void *__restrict__ out, uint16_t *__restrict__ pool, int H, int W, int CO,
                                           int ostride, int ooff, int relu, int f32_nchw, int vec, int n, int y0,
                                           int x0, int cob)
{
    constexpr int GR = 32 / TC, WC = 4 / WY, TR = WY * MT * GR, kOut = TR * TC * 4 * WC;
    const int tid = int(threadIdx.x), lane = tid % 64, wave = tid / 64, m = lane % 32, hk = lane / 32;
    const int wy = wave % WY, wc = wave / WY, co0 = cob + 32 * wc;
    // lane holds D[channel 8 (j/4) + 4 hk + j%4][pixel m] of each 32x32 tile
    float bv[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int co = co0 + 8 * (j / 4) + 4 * hk + j % 4;
        bv[j] = bias && co < CO ? bias[co] : 0.0f;
    }
    const auto value = [&](int t, int j) {
        const float v = acc[t][j] + bv[j];
        return relu ? __builtin_fmaxf(v, 0.0f) : v;
    };
    if (f32_nchw) {
        const int x = x0 + m % TC;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const int y = y0 + (wy * MT + t) * GR + m / TC;
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int co = co0 + 8 * (j / 4) + 4 * hk + j % 4;
                if (co < CO && y < H && x < W)
                    static_cast<float *>(out)[((int64_t(n) * CO + co) * H + y) * W + x] = value(t, j);
            }
        }
        return;
    }
    // slot 4 p + group of each of the WC channel blocks
    __syncthreads();
    uint2 *const so = reinterpret_cast<uint2 *>(sh + wc * (TR * TC * 4));
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int p = (wy * MT + t) * 32 + m;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            so[(4 * p + turn<4>(q, p)) * 2 + hk] = make_uint2(pack2(value(t, 4 * q), value(t, 4 * q + 1)),
                                                              pack2(value(t, 4 * q + 2), value(t, 4 * q + 3)));
        }
    }
    __syncthreads();
    uint16_t *const o = static_cast<uint16_t *>(out);
    if (vec) {
        for (int e = tid; e < kOut; e += 256) {
            const int b = e / (TR * TC * 4), p = e / 4 % (TR * TC), g = e % 4;
            const int y = y0 + p / TC, x = x0 + p % TC, co = cob + 32 * b + 8 * g;
            if (y >= H || x >= W || co >= CO) continue;
            *reinterpret_cast<uint4 *>(o + ((int64_t(n) * H + y) * W + x) * ostride + ooff + co) =
                sh[b * (TR * TC * 4) + 4 * p + turn<4>(g, p)];
        }
    } else {
        // Where 16 bytes do not fit: one channel per access, or two where CO and
        // the output's place are even, consecutive channels in consecutive
        // lanes.  A lane keeps its channel and its column modulo 8 or 16, so that
        // the addresses only step.  (8 channels per lane, each stored alone: 4 x 79
        // x 507, 16 -> 229 channels 91 us, now 37.5; 15 x 97 x 254, 16 -> 58 57 and
        // 22.6.)
        const auto narrow = [&](auto access) {
            using A = decltype(access);
            constexpr int K = sizeof(A) / 2, L = 32 / K, P = 256 / L;  // lanes per pixel, pixels at a time
            const int c = tid % L * K, px = tid / L;
#pragma unroll
            for (int b = 0; b < WC; ++b) {
                const int co = cob + 32 * b + c;
                if (co >= CO) break;
                const A *const v =
                    reinterpret_cast<const A *>(sh + (b * (TR * TC * 4) + 4 * px + turn<4>(c / 8, px))) + c % 8 / K;
                uint16_t *d = o + ((int64_t(n) * H + y0) * W + x0 + px) * ostride + ooff + co;
                const int rows = min(TR, H - y0);
                for (int r = 0; r < rows; ++r, d += int64_t(W) * ostride)
#pragma unroll
                    for (int i = 0; i < TC / P; ++i)
                        if (x0 + px + P * i < W)
                            *reinterpret_cast<A *>(d + int64_t(P * i) * ostride) = v[(r * TC + P * i) * (32 / K)];
            }
        };
        const bool two = CO % 2 == 0 && ostride % 2 == 0 && ooff % 2 == 0 && reinterpret_cast<uintptr_t>(out) % 4 == 0;
        if (two)
            narrow(uint32_t{});
        else
            narrow(uint16_t{});
    }
    if (!pool) return;
    for (int e = tid; e < kOut / 4; e += 256) {
        const int b = e / (TR * TC), q = e / 4 % (TR * TC / 4), g = e % 4;
        const int py = q / (TC / 2), px = q % (TC / 2), p = 2 * py * TC + 2 * px;
        const int y = y0 / 2 + py, x = x0 / 2 + px, co = cob + 32 * b + 8 * g;
        if (y >= H / 2 || x >= W / 2 || co >= CO) continue;
        const uint4 *const t = sh + b * (TR * TC * 4);
        *reinterpret_cast<uint4 *>(pool + ((int64_t(n) * (H / 2) + y) * (W / 2) + x) * CO + co) =
            average4(t[4 * p + turn<4>(g, p)], t[4 * (p + 1) + turn<4>(g, p + 1)],
                     t[4 * (p + TC) + turn<4>(g, p + TC)], t[4 * (p + TC + 1) + turn<4>(g, p + TC + 1)]);
    }
}

// Every sum takes its products in one order, 16 input channels after
// another and tap after tap, whatever the tile.  A plain tile (one 32-pixel
// operand read per product, weights and pixels through LDS) was bound by
// LDS reads: 2 KB per product and wave, twice what LDS gives in the 32 cycles
// of a product.  Here a wave takes MT groups of rows and holds the 9 taps'
// weights of 16 channels in registers, so that a row read once serves as the
// upper, middle and lower row of three groups: 0.5 KB per product.  The
// input goes from memory straight to LDS; two or three blocks on a CU hide
// one another's waits.  40 cases on 128 x 512: 384 -> 128 channels 210 to
// 127 us (1,140 TFLOP/s), 256 -> 256 81 to 52 us, 32 -> 32 (bound by memory,
// 336 MB) 153 to 97 us; the whole network 2.20 to 1.13 ms.
//
// 3x3 convolution, padding 1, NHWC bf16.  Input channels [0, C0) come from
// in0 at half the resolution (nearest upsampling), the following C1 from in1;
// wp: [CIP/8][9][COP] groups of 8 input channels.  Output channel co < CO of
// pixel (n, y, x): bf16 at out[((n H + y) W + x) ostride + ooff + co], or with
// f32_nchw FP32 at out[((n CO + co) H + y) W + x]; with pool also the 2x2
// average of the bf16 values at pool[((n H/2 + y/2) W/2 + x/2) CO + co].
template <int MT, int WY, int TC, int KC>
__global__ __launch_bounds__(256, MT == 4 ? 3 : 4) void k_conv3_bf16(const uint4 *__restrict__ in0, int C0,
                                                    const uint4 *__restrict__ in1, int C1,
                                                    const uint4 *__restrict__ wp, const float *__restrict__ bias,
                                                    void *__restrict__ out, uint16_t *__restrict__ pool, int H, int W,
                                                    int CO, int COP, int ostride, int ooff, int relu, int f32_nchw,
                                                    int vec, uint32_t ntx, uint32_t nty, uint32_t ncob)
{
    constexpr int G = KC / 8, GR = 32 / TC, WC = 4 / WY;
    constexpr int TR = WY * MT * GR, IR = TR + 2, IC = TC + 2, NPX = IR * IC;
    constexpr int NI = (NPX * G + 255) / 256;
    constexpr int kIn = NPX * G, kOut = TR * TC * 4 * WC;
    __shared__ uint4 sh[kIn > kOut ? kIn : kOut];
    const int tid = int(threadIdx.x), lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int m = lane % 32, hk = lane / 32;  // operand row / column and K half
    const int wy = wave % WY, wc = wave / WY;
    uint32_t blk = xcd_run(blockIdx.x, gridDim.x);
    const int cob = int(blk % ncob) * (32 * WC);
    blk /= ncob;
    const int x0 = int(blk % ntx) * TC;
    blk /= ntx;
    const int y0 = int(blk % nty) * TR, n = int(blk / nty);
    const int co0 = cob + 32 * wc;

    // staging, straight to LDS in 16-byte slots (slot e of the block is lane
    // e % 64's of its wave's load e / 256); slots outside the image stay
    // zero.  A slot's pixel is kept as row and column of the tile, -1 where
    // there is nothing to load.
    int at[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int e = tid + 256 * i, p = e / G, r = p / IC, c = p % IC;
        const int yy = y0 + r - 1, xx = x0 + c - 1;
        const bool ok = e < kIn && yy >= 0 && yy < H && xx >= 0 && xx < W;
        at[i] = ok ? r << 8 | c : -1;
        if (e < kIn && !ok) sh[e] = make_uint4(0u, 0u, 0u, 0u);
    }
    const uint4 *const t1 = in1 + ((int64_t(n) * H + y0) * W + x0) * (C1 / 8);
    const uint4 *const t0 = C0 ? in0 + ((int64_t(n) * (H / 2) + y0 / 2) * (W / 2) + x0 / 2) * (C0 / 8) : nullptr;
    int pa[3];  // the lane's pixel operand of tap column kx, row 0, first group
#pragma unroll
    for (int kx = 0; kx < 3; ++kx)
        pa[kx] = ((wy * MT * GR + m / TC) * IC + m % TC + kx) * G + turn<G>(hk, m % TC + kx);
    f32x16 acc[MT] = {};
    const int CIP = C0 + C1;
    for (int c0 = 0; c0 < CIP; c0 += KC) {
        __syncthreads();  // the previous channels have been multiplied
        const auto stage = [&](const uint4 *base, int stride, int half, int w) {
#pragma unroll
            for (int i = 0; i < NI; ++i)
                if (at[i] >= 0) {
                    const int r = (at[i] >> 8) - 1 >> half, c = (at[i] & 255) - 1 >> half;
                    const int g = turn<G>(tid % G, at[i] & 255);
                    __builtin_amdgcn_global_load_lds(
                        (const __attribute__((address_space(1))) void *)(base + int64_t(r * w + c) * stride + g),
                        (__attribute__((address_space(3))) void *)(sh + 256 * i + 64 * wave), 16, 0, 0);
                }
        };
        if (c0 < C0)
            stage(t0 + c0 / 8, C0 / 8, 1, W / 2);
        else
            stage(t1 + (c0 - C0) / 8, C1 / 8, 0, W);
        // the weights of 16 channels: every lane its output channel's 8 of K
        bf16x8 wf[9];
        auto weights = [&](int c) {
            const uint4 *const p = wp + (int64_t(c / 8 + hk) * 9) * COP + co0 + m;
#pragma unroll
            for (int t = 0; t < 9; ++t) wf[t] = __builtin_bit_cast(bf16x8, p[int64_t(t) * COP]);
        };
        weights(c0);
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's slots are in LDS
        __syncthreads();
#pragma unroll
        for (int cc = 0; cc < KC / 16; ++cc) {
            if (cc > 0) weights(c0 + 16 * cc);
            // input rows in order; each serves the (up to three) groups of
            // output rows that it is the upper, middle or lower row of, so
            // every sum takes its taps in order
#pragma unroll
            for (int s = 0; s < (MT - 1) * GR + 3; ++s)
#pragma unroll
                for (int kx = 0; kx < 3; ++kx) {
                    const bf16x8 a = __builtin_bit_cast(bf16x8, sh[(pa[kx] ^ 2 * cc) + s * IC * G]);
#pragma unroll
                    for (int ky = 0; ky < 3; ++ky)
                        if ((s - ky) % GR == 0 && s - ky >= 0 && (s - ky) / GR < MT)
                            acc[(s - ky) / GR] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[3 * ky + kx], a,
                                                                                         acc[(s - ky) / GR], 0, 0, 0);
                }
        }
    }
    conv_store<MT, WY, TC>(acc, sh, bias, out, pool, H, W, CO, ostride, ooff, relu, f32_nchw, vec, n, y0, x0, cob);
}

// The same for few tiles (a block or less per CU), where the time is that of
// one block's chain of chunks: input and weights of the next three chunks
// are on their way to LDS while one is multiplied.  Every wave issues the
// same number of loads per chunk (a slot with nothing to load takes zeros),
// so it can wait for the oldest chunk alone.
__device__ const uint4 zero_slot = {0u, 0u, 0u, 0u};
template <int TC, int KC>
__global__ __launch_bounds__(256) void k_conv3_bf16_deep(const uint4 *__restrict__ in0, int C0,
                                                         const uint4 *__restrict__ in1, int C1,
                                                         const uint4 *__restrict__ wp, const float *__restrict__ bias,
                                                         void *__restrict__ out, uint16_t *__restrict__ pool, int H,
                                                         int W, int CO, int COP, int ostride, int ooff, int relu,
                                                         int f32_nchw, int vec, uint32_t ntx, uint32_t nty,
                                                         uint32_t ncob)
{
    constexpr int G = KC / 8, GR = 32 / TC, TR = 4 * GR, IR = TR + 2, IC = TC + 2;
    constexpr int kIn = IR * IC * G, NI = (kIn + 255) / 256, kW = 9 * G * 32, NW = (kW + 255) / 256;
    constexpr int kBuf = (NI + NW) * 256, ND = 4;
    __shared__ uint4 sh[ND * kBuf];
    const int tid = int(threadIdx.x), lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int m = lane % 32, hk = lane / 32;
    uint32_t blk = xcd_run(blockIdx.x, gridDim.x);
    const int co0 = int(blk % ncob) * 32;
    blk /= ncob;
    const int x0 = int(blk % ntx) * TC;
    blk /= ntx;
    const int y0 = int(blk % nty) * TR, n = int(blk / nty);
    const uint4 *const t1 = in1 + ((int64_t(n) * H + y0) * W + x0) * (C1 / 8);
    const uint4 *const t0 = C0 ? in0 + ((int64_t(n) * (H / 2) + y0 / 2) * (W / 2) + x0 / 2) * (C0 / 8) : nullptr;
    const auto put = [&](const uint4 *a, uint4 *d) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)a,
                                         (__attribute__((address_space(3))) void *)d, 16, 0, 0);
    };
    const auto stage = [&](int c0, int buf) {
        uint4 *const d = sh + buf * kBuf + 64 * wave;
        const bool low = c0 < C0;
        const uint4 *const base = low ? t0 + c0 / 8 : t1 + (c0 - C0) / 8;
        const int stride = (low ? C0 : C1) / 8, w = low ? W / 2 : W, half = low ? 1 : 0;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int e = tid + 256 * i, p = e / G, r = p / IC - 1, c = p % IC - 1;
            const bool ok = e < kIn && unsigned(y0 + r) < unsigned(H) && unsigned(x0 + c) < unsigned(W);
            const int64_t o = int64_t((r >> half) * w + (c >> half)) * stride + turn<G>(tid % G, c + 1);
            put(ok ? base + o : &zero_slot, d + 256 * i);
        }
        const uint4 *const wb = wp + int64_t(c0 / 8) * 9 * COP + co0;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int e = tid + 256 * i;
            put(e < kW ? wb + int64_t(e / 32) * COP + e % 32 : &zero_slot, d + 256 * (NI + i));
        }
    };
    int pa[3];
#pragma unroll
    for (int kx = 0; kx < 3; ++kx)
        pa[kx] = ((wave * GR + m / TC) * IC + m % TC + kx) * G + turn<G>(hk, m % TC + kx);
    f32x16 acc[1] = {};
    const int nst = (C0 + C1) / KC;
#pragma unroll
    for (int k = 0; k < ND - 1; ++k)
        if (k < nst) stage(k * KC, k);
    for (int st = 0; st < nst; ++st) {
        // this chunk has arrived once only the later ones' loads are out
        const int later = min(ND - 2, nst - 1 - st);
        static_assert(ND == 4 && 2 * (NI + NW) < 64, "the counts below");
        constexpr int v2 = 2 * (NI + NW), v1 = NI + NW;
        if (later == 2)
            __builtin_amdgcn_s_waitcnt(0x0f70 | (v2 & 15) | (v2 >> 4) << 14);
        else if (later == 1)
            __builtin_amdgcn_s_waitcnt(0x0f70 | (v1 & 15) | (v1 >> 4) << 14);
        else
            __builtin_amdgcn_s_waitcnt(0x0f70);
        // for every wave; and the previous chunk has been multiplied.  (Not
        // __syncthreads(), whose fence waits for the later chunks too.)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (st + ND - 1 < nst) stage((st + ND - 1) * KC, (st + ND - 1) % ND);
        const uint4 *const si = sh + st % ND * kBuf, *const sw = si + 256 * NI;
        // operands read three products ahead
        constexpr int NP = KC / 16 * 9, AH = 3;
        bf16x8 a[AH + 1], b[AH + 1];
        const auto fetch = [&](int q) {
            const int cc = q / 9, t = q % 9;
            a[q % (AH + 1)] = __builtin_bit_cast(bf16x8, sw[((2 * cc + hk) * 9 + t) * 32 + m]);
            b[q % (AH + 1)] = __builtin_bit_cast(bf16x8, si[(pa[t % 3] ^ 2 * cc) + t / 3 * IC * G]);
        };
#pragma unroll
        for (int q = 0; q < AH; ++q) fetch(q);
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * AH, 0);
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            if (q + AH < NP) fetch(q + AH);
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[q % (AH + 1)], b[q % (AH + 1)], acc[0], 0, 0, 0);
            if (q + AH < NP) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
    }
    __syncthreads();
    conv_store<1, 4, TC>(acc, sh, bias, out, pool, H, W, CO, ostride, ooff, relu, f32_nchw, vec, n, y0, x0, co0);
}

// x [N][C][H][W] FP32 -> y [N][H][W][CP] bf16, channels C..CP-1 zero; K
// channels per thread (8 where CP is a multiple of 8: one 16-byte store)
template <int K>
__global__ __launch_bounds__(256) void k_pack_in(const float *__restrict__ x, uint16_t *__restrict__ y, int C, int CP,
                                                 int64_t hw, int64_t total)
{
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= total) return;
    const int cg = CP / K;
    const int64_t n = i / (hw * cg), j = i - n * hw * cg;
    const int c = int(j / hw) * K;  // a wave reads consecutive pixels of a channel
    const int64_t r = j - (c / K) * hw;
    uint16_t v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = c + k < C ? to_bf16(x[(n * C + c + k) * hw + r]) : uint16_t(0);
    uint16_t *const o = y + (n * hw + r) * CP + c;
    if constexpr (K == 8)
        *reinterpret_cast<uint4 *>(o) =
            make_uint4(v[0] | uint32_t(v[1]) << 16, v[2] | uint32_t(v[3]) << 16, v[4] | uint32_t(v[5]) << 16,
                       v[6] | uint32_t(v[7]) << 16);
    else
        *o = v[0];
}

// w [CO][CI][3][3] FP32 -> wp [CIP/8][9][COP][8] bf16, zero outside CO x CI
__global__ void k_pack_w(const float *__restrict__ w, uint16_t *__restrict__ wp, int CI, int CO, int COP,
                         int64_t total)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int j = int(i % 8), co = int((i / 8) % COP), t = int((i / (8 * int64_t(COP))) % 9);
    const int ci = int(i / (72 * int64_t(COP))) * 8 + j;
    wp[i] = (co < CO && ci < CI) ? to_bf16(w[(int64_t(co) * CI + ci) * 9 + t]) : uint16_t(0);
}

// 2x2 average pool of channels [coff, coff + 8 C8) of in [N][2h][2w][8 cs8]
// into out [N][h][w][8 C8]; one thread per 8 channels
__global__ void k_pool2_bf16(const uint4 *__restrict__ in, uint4 *__restrict__ out, int h, int w, int cs8, int coff8,
                             int C8, int64_t total)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int g = int(i % C8);
    const int64_t p = i / C8;
    const int x = int(p % w), y = int((p / w) % h);
    const int64_t n = p / (int64_t(w) * h);
    const int64_t b = ((n * 2 * h + 2 * y) * 2 * w + 2 * x) * cs8 + coff8 + g;
    out[i] = average4(in[b], in[b + cs8], in[b + 2 * int64_t(w) * cs8], in[b + (2 * int64_t(w) + 1) * cs8]);
}

// nearest 2x upsample of in [N][h][w][8 C8] into channels [coff, coff + 8 C8)
// of out [N][2h][2w][8 ct8]
__global__ void k_up2_bf16(const uint4 *__restrict__ in, uint4 *__restrict__ out, int h, int w, int ct8, int coff8,
                           int C8, int64_t total)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int g = int(i % C8);
    const int64_t p = i / C8;
    const int X = int(p % (2 * w)), Y = int((p / (2 * w)) % (2 * h));
    const int64_t n = p / (int64_t(4) * w * h);
    out[p * ct8 + coff8 + g] = in[((n * h + Y / 2) * w + X / 2) * C8 + g];
}

inline unsigned blocks(int64_t n) { return unsigned((n + 255) / 256); }

// the buffers of a pooling or upsampling call take 8- and 16-byte accesses
inline bool vec_ok(int w, std::initializer_list<const void *> ptrs)
{
    uintptr_t bits = 0;
    for (const void *p : ptrs) bits |= reinterpret_cast<uintptr_t>(p);
    return w % 2 == 0 && bits % 16 == 0;
}
template <class K, class... Args>
int launch_low_res(bool wide, K aligned, K plain, int N, int C, int h, int w, void *stream, Args... args)
{
    LowRes g{N, C, h, w, 0, {}, {}, {}};
    const int per_row = wide ? w / 2 : w;
    const int64_t rows = int64_t(N) * C * h;
    if (rows <= 0x7fffffff / per_row) {
        g.items = uint32_t(rows * per_row);
        g.per_row.init(uint32_t(per_row));
        g.rows.init(uint32_t(h));
        g.chans.init(uint32_t(C));
    }
    const unsigned nb = g.items ? blocks(g.items) : unsigned(std::min<int64_t>((rows + 3) / 4, int64_t(1) << 20));
    hipLaunchKernelGGL(wide ? aligned : plain, dim3(nb), dim3(256), 0, (hipStream_t)stream, args..., g);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// the convolution's tile for these sizes and its launch
template <bool DGRAD>
int launch_conv(const float *in, const float *w, const float *bias, float *out, int ototal, const float *gate,
                int gtotal, int N, int CI, int CO, int H, int W, int relu, hipStream_t stream)
{
    // The largest tile that still gives every CU two blocks (its operands are
    // reused most: 8 x 32 pixels for 64 channels 118 TFLOP/s on the deep
    // layers of a batch of 8, for 32 channels 100); a batch of one gets the
    // smallest.  Rows of at most 16 pixels take the 16-column tile.
    const auto run = [&](auto kernel, int rows, int cols, int bn, bool always) {
        const int64_t tx = (int64_t(W) + cols - 1) / cols, ty = (int64_t(H) + rows - 1) / rows, tc = (CO + bn - 1) / bn;
        const int64_t nb = tx * ty * tc * N;
        if (nb < 512 && !always) return 1;  // too few blocks to give every CU two: smaller tiles
        if (nb > 0x7fffffff) return -2;
        hipLaunchKernelGGL(kernel, dim3(unsigned(nb)), dim3(256), 0, stream, in, w, bias, out, ototal, gate,
                           gtotal, CI, CO, H, W, relu, uint32_t(tx), uint32_t(ty), uint32_t(tc));
        return hipGetLastError() == hipSuccess ? 0 : -2;
    };
    const auto tile = [&](auto few) {
        constexpr bool F = decltype(few)::value;
        if (W <= 16) return run(k_conv3<1, 1, 16, DGRAD, F>, 8, 16, 32, true);
        int rc = CO > 32 ? run(k_conv3<2, 2, 32, DGRAD, F>, 8, 32, 64, false) : 1;
        if (rc > 0) rc = run(k_conv3<2, 1, 32, DGRAD, F>, 8, 32, 32, false);
        return rc <= 0 ? rc : run(k_conv3<1, 1, 32, DGRAD, F>, 4, 32, 32, true);
    };
    return CI <= 6 ? tile(std::true_type{}) : tile(std::false_type{});
}

// weight gradient: the tiles' sums to `work` and from there to dw in tile
// order, or (work == nullptr) to dw with atomics; db: the bias gradient too.
int launch_dw(const float *in, const float *dout, float *dw, float *db, float *work, int N, int CI, int CO, int H,
              int W, hipStream_t s)
{
    const int64_t tiles = int64_t((W + TS - 1) / TS) * ((H + TS - 1) / TS), n = int64_t(CO) * CI * 9;
    // blocks of 32 x 32 channels share their staged pixels most; where they
    // leave CUs without a block, smaller ones, whose waves share the taps
    // (64 -> 128, 8 x 32 x 128: 108 us with 128 blocks, 69 us with 256),
    // and 16 x 16 as the last resort
    const auto pairs = [&](int gco, int gci) {
        return int64_t((CO + 16 * gco - 1) / (16 * gco)) * ((CI + 16 * gci - 1) / (16 * gci));
    };
    int gco = 1, gci = 1;
    if (CO > 16 && CI > 16 && tiles * pairs(2, 2) >= 256)
        gco = gci = 2;
    else if (CO > 16 && tiles * pairs(2, 1) >= 256)
        gco = 2;
    else if (CI > 16 && tiles * pairs(1, 2) >= 256)
        gci = 2;
    const dim3 grid(unsigned(tiles), unsigned(pairs(gco, gci) + (db ? 1 : 0)));
    const auto kernel = gco == 2 ? (gci == 2 ? k_conv3_dw<2, 2> : k_conv3_dw<2, 1>)
                                 : (gci == 2 ? k_conv3_dw<1, 2> : k_conv3_dw<1, 1>);
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, in, dout, dw, N, CI, CO, H, W, work, db);
    if (hipGetLastError() != hipSuccess) return -2;
    if (!work) return 0;
    hipLaunchKernelGGL(k_dw_reduce, dim3(unsigned((n + 63) / 64)), dim3(64), 0, s, work, dw, tiles, n);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace imexlb_nn

using namespace imexlb_nn;

#define NN_LAUNCH(...)                                                  \
    do {                                                                \
        hipLaunchKernelGGL(__VA_ARGS__);                                \
        return hipGetLastError() == hipSuccess ? 0 : -2;                \
    } while (0)

extern "C" {

int imexlb_nn_conv3x3(const float *in, const float *w, const float *bias, float *out, int N, int CI, int CO, int H,
                      int W, int relu, void *stream)
{
    if (!in || !w || !out || N <= 0 || CI <= 0 || CO <= 0 || H <= 0 || W <= 0) return -1;
    return launch_conv<false>(in, w, bias, out, CO, nullptr, 0, N, CI, CO, H, W, relu, (hipStream_t)stream);
}

int imexlb_nn_conv3x3_into(const float *in, const float *w, const float *bias, float *out, int ototal, int ooff, int N,
                           int CI, int CO, int H, int W, int relu, void *stream)
{
    if (!in || !w || !out || N <= 0 || CI <= 0 || CO <= 0 || H <= 0 || W <= 0 || ooff < 0 || ooff + CO > ototal)
        return -1;
    return launch_conv<false>(in, w, bias, out + int64_t(ooff) * H * W, ototal, nullptr, 0, N, CI, CO, H, W, relu,
                              (hipStream_t)stream);
}

int imexlb_nn_conv3x3_dgrad(const float *dz, const float *w, const float *gate, int gtotal, int goff, float *dx, int N,
                            int CI, int CO, int H, int W, void *stream)
{
    if (!dz || !w || !dx || N <= 0 || CI <= 0 || CO <= 0 || H <= 0 || W <= 0 ||
        (gate && (goff < 0 || goff + CI > gtotal)))
        return -1;
    return launch_conv<true>(dz, w, nullptr, dx, CI, gate ? gate + int64_t(goff) * H * W : nullptr, gtotal, N, CO, CI, H,
                             W, 0, (hipStream_t)stream);
}

int imexlb_nn_flip_weights(const float *w, float *wt, int CI, int CO, void *stream)
{
    if (!w || !wt || CI <= 0 || CO <= 0) return -1;
    NN_LAUNCH(k_flip, dim3(blocks(int64_t(CO) * CI * 9)), dim3(256), 0, (hipStream_t)stream, w, wt, CI, CO);
}

int imexlb_nn_conv3x3_dw(const float *in, const float *dout, float *dw, int N, int CI, int CO, int H, int W,
                         void *stream)
{
    if (!in || !dout || !dw || N <= 0 || CI <= 0 || CO <= 0 || H <= 0 || W <= 0) return -1;
    return launch_dw(in, dout, dw, nullptr, nullptr, N, CI, CO, H, W, (hipStream_t)stream);
}

int64_t imexlb_nn_conv3x3_dw_work(int CI, int CO, int H, int W)
{
    if (CI <= 0 || CO <= 0 || H <= 0 || W <= 0) return -1;
    return int64_t((W + TS - 1) / TS) * ((H + TS - 1) / TS) * CO * CI * 9;
}

int imexlb_nn_conv3x3_dw_ordered(const float *in, const float *dout, float *dw, float *work, int64_t work_floats,
                                 int N, int CI, int CO, int H, int W, void *stream)
{
    if (!in || !dout || !dw || !work || N <= 0 || CI <= 0 || CO <= 0 || H <= 0 || W <= 0) return -1;
    const int64_t tiles = int64_t((W + TS - 1) / TS) * ((H + TS - 1) / TS);
    const int64_t n = int64_t(CO) * CI * 9;
    if (work_floats < tiles * n) return -1;
    return launch_dw(in, dout, dw, nullptr, work, N, CI, CO, H, W, (hipStream_t)stream);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// The ordered weight gradient without a caller workspace: the per-tile sums
// go to `scratch`, a device array of the library that every GPU it runs on
// holds until the process ends.  Host code reaches it only through the
// address hipGetSymbolAddress gives on each device (the array's name is a
// host-side stand-in).  Nothing in it needs to start at zero: k_conv3_dw
// writes every partial that k_dw_reduce then reads.  Calls that overlap on
// one GPU share the array and race.
constexpr int64_t kScratchFloats = int64_t(8) << 20;  // 8 Mi floats, 32 MiB
static __device__ __align__(256) float scratch[kScratchFloats];

namespace {

constexpr int kMaxDevices = 64;
std::mutex scratch_mu;
float *scratch_dev[kMaxDevices] = {};

// this device's copy of scratch (the caller's current device), looked up on
// the first call on the device; nullptr with the error text set otherwise
float *scratch_here()
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        imexlb::fail(IMEXLB_E_HIP, std::string("no usable current device: ") + hipGetErrorString(e));
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (!scratch_dev[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            imexlb::fail(IMEXLB_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
            return nullptr;
        }
        scratch_dev[dev] = static_cast<float *>(p);
    }
    return scratch_dev[dev];
}

}  // namespace

extern "C" {

int imexlb_nn_conv3x3_dw_ordered_noalloc(const float *in, const float *dout, float *dw, int N, int CI, int CO,
                                         int H, int W, void *stream)
{
    if (!in || !dout || !dw || N <= 0 || CI <= 0 || CO <= 0 || H <= 0 || W <= 0) return -1;
    const int64_t tiles = int64_t((W + TS - 1) / TS) * ((H + TS - 1) / TS);
    const int64_t n = int64_t(CO) * CI * 9;
    if (tiles * n > kScratchFloats) {
        imexlb::fail(IMEXLB_E_ARG, "weight gradient needs " + std::to_string(tiles * n) +
                                       " floats of partial sums; the library's scratch holds " +
                                       std::to_string(kScratchFloats));
        return -1;
    }
    float *work = scratch_here();
    if (!work) return -2;
    return launch_dw(in, dout, dw, nullptr, work, N, CI, CO, H, W, (hipStream_t)stream);
}

int imexlb_nn_conv3x3_grads(const float *in, const float *dout, float *dw, float *db, float *work, int64_t work_floats,
                            int N, int CI, int CO, int H, int W, void *stream)
{
    if (!in || !dout || !dw || !db || !work || N <= 0 || CI <= 0 || CO <= 0 || H <= 0 || W <= 0) return -1;
    if (work_floats < imexlb_nn_conv3x3_dw_work(CI, CO, H, W)) return -1;
    return launch_dw(in, dout, dw, db, work, N, CI, CO, H, W, (hipStream_t)stream);
}

int imexlb_nn_bias_grad(const float *dout, float *db, int N, int C, int H, int W, void *stream)
{
    if (!dout || !db || N <= 0 || C <= 0 || H <= 0 || W <= 0) return -1;
    NN_LAUNCH(k_bias_grad, dim3(unsigned(C)), dim3(256), 0, (hipStream_t)stream, dout, db, N, C, int64_t(H) * W);
}

int imexlb_nn_relu_bwd(const float *out, const float *dout, float *dz, int64_t n, void *stream)
{
    if (!out || !dout || !dz || n <= 0) return -1;
    NN_LAUNCH(k_relu_bwd, dim3(blocks(n)), dim3(256), 0, (hipStream_t)stream, out, dout, dz, n);
}

int imexlb_nn_pool2_from(const float *in, int Ctot, int coff, float *out, int N, int C, int h, int w, void *stream)
{
    if (!in || !out || N <= 0 || C <= 0 || h <= 0 || w <= 0 || coff < 0 || coff + C > Ctot) return -1;
    in += int64_t(coff) * 4 * h * w;
    return launch_low_res(vec_ok(w, {in, out}), k_pool2<true>, k_pool2<false>, N, C, h, w, stream, in, Ctot, out);
}

int imexlb_nn_pool2(const float *in, float *out, int N, int C, int h, int w, void *stream)
{
    return imexlb_nn_pool2_from(in, C, 0, out, N, C, h, w, stream);
}

int imexlb_nn_pool2_bwd_join(const float *dout, const float *skip, int stotal, int soff, const float *gate, int gtotal,
                             int goff, float *din, int N, int C, int h, int w, void *stream)
{
    if (!dout || !din || N <= 0 || C <= 0 || h <= 0 || w <= 0 || (skip && (soff < 0 || soff + C > stotal)) ||
        (gate && (goff < 0 || goff + C > gtotal)))
        return -1;
    const int64_t hw = int64_t(4) * h * w;
    if (skip) skip += soff * hw;
    if (gate) gate += goff * hw;
    return launch_low_res(vec_ok(w, {dout, skip, gate, din}), k_pool2_bwd<true>, k_pool2_bwd<false>, N, C, h, w, stream,
                          dout, skip, stotal, gate, gtotal, din);
}

int imexlb_nn_pool2_bwd(const float *dout, float *din, int N, int C, int h, int w, void *stream)
{
    return imexlb_nn_pool2_bwd_join(dout, nullptr, 0, 0, nullptr, 0, 0, din, N, C, h, w, stream);
}

int imexlb_nn_up2(const float *in, float *out, int N, int C, int h, int w, int Ctot, int coff, void *stream)
{
    if (!in || !out || N <= 0 || C <= 0 || h <= 0 || w <= 0 || coff < 0 || coff + C > Ctot) return -1;
    out += int64_t(coff) * 4 * h * w;
    return launch_low_res(vec_ok(w, {in, out}), k_up2<true>, k_up2<false>, N, C, h, w, stream, in, out, Ctot);
}

int imexlb_nn_up2_bwd_gate(const float *dout, int Ctot, int coff, const float *gate, int gtotal, int goff, float *din,
                           int N, int C, int h, int w, void *stream)
{
    if (!dout || !din || N <= 0 || C <= 0 || h <= 0 || w <= 0 || coff < 0 || coff + C > Ctot ||
        (gate && (goff < 0 || goff + C > gtotal)))
        return -1;
    dout += int64_t(coff) * 4 * h * w;
    if (gate) gate += int64_t(goff) * h * w;
    return launch_low_res(vec_ok(w, {dout, gate, din}), k_up2_bwd<true>, k_up2_bwd<false>, N, C, h, w, stream, dout, Ctot,
                          gate, gtotal, din);
}

int imexlb_nn_up2_bwd(const float *dout, float *din, int N, int C, int h, int w, int Ctot, int coff, void *stream)
{
    return imexlb_nn_up2_bwd_gate(dout, Ctot, coff, nullptr, 0, 0, din, N, C, h, w, stream);
}

int imexlb_nn_copy_channels(const float *src, int sctot, int scoff, float *dst, int dctot, int dcoff, int N, int C,
                            int H, int W, int accumulate, void *stream)
{
    if (!src || !dst || N <= 0 || C <= 0 || H <= 0 || W <= 0 || scoff < 0 || dcoff < 0 || scoff + C > sctot ||
        dcoff + C > dctot)
        return -1;
    const int64_t HW = int64_t(H) * W;
    NN_LAUNCH(k_copy_ch, dim3(blocks(int64_t(N) * C * HW)), dim3(256), 0, (hipStream_t)stream, src, sctot, scoff,
              dst, dctot, dcoff, N, C, HW, accumulate);
}

int imexlb_nn_mse(const float *pred, const float *target, float *grad, int64_t n, float *loss, void *stream)
{
    if (!pred || !target || n <= 0) return -1;
    NN_LAUNCH(k_mse, dim3(unsigned(std::min<int64_t>((n + 1023) / 1024, kMseBlocks))), dim3(1024), 0, (hipStream_t)stream, pred, target, grad, n, loss);
}

int imexlb_nn_adam(float *w, const float *g, float *m, float *v, int64_t n, float lr, float b1, float b2, float eps,
                   int step, void *stream)
{
    if (!w || !g || !m || !v || n <= 0 || step < 1) return -1;
    float c1 = 1.0f, c2 = 1.0f, p1 = 1.0f, p2 = 1.0f;
    for (int t = 0; t < step && t < 100000; ++t) {
        p1 *= b1;
        p2 *= b2;
    }
    c1 = 1.0f - p1;
    c2 = 1.0f - p2;
    NN_LAUNCH(k_adam, dim3(blocks(n)), dim3(256), 0, (hipStream_t)stream, w, g, m, v, n, lr, b1, b2, eps, c1, c2);
}

int imexlb_nn_pack_input_bf16(const float *x, uint16_t *y, int N, int C, int CP, int H, int W, void *stream)
{
    if (!x || !y || N <= 0 || C <= 0 || CP < C || H <= 0 || W <= 0) return -1;
    const int64_t hw = int64_t(H) * W;
    const bool wide = CP % 8 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
    const int64_t total = N * hw * (wide ? CP / 8 : CP);
    NN_LAUNCH(wide ? k_pack_in<8> : k_pack_in<1>, dim3(blocks(total)), dim3(256), 0, (hipStream_t)stream, x, y, C, CP,
              hw, total);
}

int imexlb_nn_pack_weights_bf16(const float *w, uint16_t *wp, int CI, int CO, int CIP, int COP, void *stream)
{
    if (!w || !wp || CI <= 0 || CO <= 0 || CIP < CI || CIP % 8 || COP < CO) return -1;
    const int64_t total = int64_t(CIP) * 9 * COP;
    NN_LAUNCH(k_pack_w, dim3(blocks(total)), dim3(256), 0, (hipStream_t)stream, w, wp, CI, CO, COP, total);
}

int imexlb_nn_conv3x3_bf16(const uint16_t *in, const uint16_t *wp, const float *bias, void *out, int N, int CIP,
                           int CO, int COP, int H, int W, int ostride, int ooff, int relu, int f32_nchw, void *stream)
{
    return imexlb_nn_conv3x3_bf16_join(nullptr, 0, in, CIP, wp, bias, out, nullptr, N, CO, COP, H, W, ostride, ooff,
                                       relu, f32_nchw, stream);
}

int imexlb_nn_conv3x3_bf16_join(const uint16_t *low, int CL, const uint16_t *in, int CI, const uint16_t *wp,
                                const float *bias, void *out, uint16_t *pool, int N, int CO, int COP, int H, int W,
                                int ostride, int ooff, int relu, int f32_nchw, void *stream)
{
    if (!in || !wp || !out || N <= 0 || N > 65535 || H <= 0 || W <= 0 || CI <= 0 || CI % 16 || CO <= 0 || COP < CO ||
        COP % 32)
        return -1;
    if (low ? CL <= 0 || CL % 16 || H % 2 || W % 2 : CL != 0) return -1;
    if (pool && (f32_nchw || H % 2 || W % 2 || CO % 8)) return -1;
    if (!f32_nchw && (ooff < 0 || ooff + CO > ostride)) return -1;
    if ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(wp) | reinterpret_cast<uintptr_t>(low) |
         reinterpret_cast<uintptr_t>(pool)) & 15)
        return -1;
    const int vec = CO % 8 == 0 && ostride % 8 == 0 && ooff % 8 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    const auto count = [&](int rows, int cols, int bn) {
        return ((int64_t(W) + cols - 1) / cols) * ((int64_t(H) + rows - 1) / rows) * ((COP + bn - 1) / bn) * N;
    };
    const auto run = [&](auto kernel, int rows, int cols, int bn) {
        if (count(rows, cols, bn) > 0x7fffffff) return -1;
        hipLaunchKernelGGL(kernel, dim3(unsigned(count(rows, cols, bn))), dim3(256), 0, (hipStream_t)stream,
                           reinterpret_cast<const uint4 *>(low), CL, reinterpret_cast<const uint4 *>(in), CI,
                           reinterpret_cast<const uint4 *>(wp), bias, out, pool, H, W, CO, COP, ostride, ooff, relu,
                           f32_nchw, vec, uint32_t((W + cols - 1) / cols), uint32_t((H + rows - 1) / rows),
                           uint32_t((COP + bn - 1) / bn));
        return hipGetLastError() == hipSuccess ? 0 : -2;
    };
    // 32 channels a chunk where the inputs allow it.  The widest tile that
    // gives every CU two blocks; for 32 output channels of few input channels
    // (bound by memory) 16 rows of 16-channel chunks, else 8 rows (40 x 128 x
    // 512, 32 -> 32 channels 93 against 100 us, 96 -> 32 245 against 229 us).
    // Below that the chain of chunks is the time: three chunks ahead (a batch
    // of one on 128 x 512: 116 us for the whole network, 137 with the plain
    // 4-row tile for the layers of one and two chunks, 223 for all).
    const bool wide = CI % 32 == 0 && CL % 32 == 0;
#define CONV_BF16(MT, WY, TC) (wide ? k_conv3_bf16<MT, WY, TC, 32> : k_conv3_bf16<MT, WY, TC, 16>)
#define CONV_BF16_DEEP(TC) (wide ? k_conv3_bf16_deep<TC, 32> : k_conv3_bf16_deep<TC, 16>)
    // Rows of at most 16 pixels: three chunks ahead up to a block per CU, and of
    // many input channels somewhat above (us, ahead and plain, blocks: 32
    // channels 6.8 and 6.7 at 208, 13.8 and 8.2 at 800; 128 7.2 and 10.2 at 208,
    // 11.6 and 11.6 at 320, 21.9 and 17.7 at 800; 512 40 and 43 at 640).
    if (W <= 16)
        return count(8, 16, 32) <= std::max<int64_t>(256, (int64_t(CL) + CI) * 5 / 2) ? run(CONV_BF16_DEEP(16), 8, 16, 32)
                                                                                 : run(CONV_BF16(1, 4, 16), 8, 16, 32);
    if (COP % 64 == 0 && count(8, 32, 64) >= 512) return run(CONV_BF16(4, 2, 32), 8, 32, 64);
    if (CL + CI <= 32 && count(16, 32, 32) >= 512) return run(k_conv3_bf16<4, 4, 32, 16>, 16, 32, 32);
    if (count(8, 32, 32) >= 512) return run(CONV_BF16(2, 4, 32), 8, 32, 32);
    // (more blocks than CUs, of one or two chunks, or of up to eight where 8 rows
    // cover no more than 4: 40 x 64 x 24, 32 -> 16 channels 11.0 and, plain, 7.1
    // us; 8 x 128 x 48, 64 -> 32 10.1 and 8.8; 32 x 5 x 41, 96 -> 210 20.2 and 11.6)
    if (wide && count(4, 32, 32) > 256 &&
        (CL + CI <= 64 || (CL + CI <= 256 && 2 * count(8, 32, 32) <= count(4, 32, 32))))
        return run(CONV_BF16(2, 4, 32), 8, 32, 32);
    return run(CONV_BF16_DEEP(32), 4, 32, 32);
#undef CONV_BF16_DEEP
#undef CONV_BF16
}

int imexlb_nn_pool2_bf16(const uint16_t *in, uint16_t *out, int N, int C, int h, int w, int cstride, int coff,
                         void *stream)
{
    if (!in || !out || N <= 0 || C <= 0 || h <= 0 || w <= 0 || C % 8 || cstride % 8 || coff % 8 || coff < 0 ||
        coff + C > cstride)
        return -1;
    if ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) return -1;
    const int64_t total = int64_t(N) * h * w * (C / 8);
    NN_LAUNCH(k_pool2_bf16, dim3(blocks(total)), dim3(256), 0, (hipStream_t)stream,
              reinterpret_cast<const uint4 *>(in), reinterpret_cast<uint4 *>(out), h, w, cstride / 8, coff / 8, C / 8,
              total);
}

int imexlb_nn_up2_bf16(const uint16_t *in, uint16_t *out, int N, int C, int h, int w, int Ctot, int coff,
                       void *stream)
{
    if (!in || !out || N <= 0 || C <= 0 || h <= 0 || w <= 0 || C % 8 || Ctot % 8 || coff % 8 || coff < 0 ||
        coff + C > Ctot)
        return -1;
    if ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) return -1;
    const int64_t total = int64_t(N) * 4 * h * w * (C / 8);
    NN_LAUNCH(k_up2_bf16, dim3(blocks(total)), dim3(256), 0, (hipStream_t)stream,
              reinterpret_cast<const uint4 *>(in), reinterpret_cast<uint4 *>(out), h, w, Ctot / 8, coff / 8, C / 8,
              total);
}

}  // extern "C"
