/* nn_chain.c -- the FP32 convolution and its weight gradient as the plain
 * loops whose sums the kernels reproduce bit for bit: one fused multiply-add
 * after another, in the order of the indices. */
#include <math.h>
#include <stdint.h>
#include <stdlib.h>

/* out[n][co][y][x] = bias[co] + the sum over ci and the taps, k = 9 ci + tap */
void conv_chain(const float *in, const float *w, const float *bias, float *out, int N, int CI, int CO, int H, int W)
{
    const int64_t PW = W + 2, PP = (int64_t)(H + 2) * PW;
    float *pad = calloc((size_t)(N * CI) * (size_t)PP, sizeof(float));
    for (int64_t c = 0; c < (int64_t)N * CI; ++c)
        for (int y = 0; y < H; ++y)
            for (int x = 0; x < W; ++x) pad[c * PP + (y + 1) * PW + x + 1] = in[(c * H + y) * W + x];
#pragma omp parallel for collapse(2)
    for (int n = 0; n < N; ++n)
        for (int co = 0; co < CO; ++co)
            for (int y = 0; y < H; ++y) {
                float *o = out + (((int64_t)n * CO + co) * H + y) * W;
                for (int x = 0; x < W; ++x) o[x] = 0.0f;
                for (int ci = 0; ci < CI; ++ci)
                    for (int t = 0; t < 9; ++t) {
                        const float v = w[((int64_t)co * CI + ci) * 9 + t];
                        const float *p = pad + ((int64_t)n * CI + ci) * PP + (y + t / 3) * PW + t % 3;
                        for (int x = 0; x < W; ++x) o[x] = fmaf(v, p[x], o[x]);
                    }
                for (int x = 0; x < W; ++x) o[x] += bias[co];
            }
    free(pad);
}

/* dw[co][ci][tap]: within a 16 x 16 tile of pixels image after image and row
 * after row, then the tiles' sums in order */
void dw_chain(const float *in, const float *g, float *dw, int N, int CI, int CO, int H, int W)
{
#pragma omp parallel for collapse(2)
    for (int co = 0; co < CO; ++co)
        for (int ci = 0; ci < CI; ++ci)
            for (int t = 0; t < 9; ++t) {
                float sum = 0.0f;
                for (int y0 = 0; y0 < H; y0 += 16)
                    for (int x0 = 0; x0 < W; x0 += 16) {
                        float s = 0.0f;
                        for (int n = 0; n < N; ++n)
                            for (int y = y0; y < y0 + 16 && y < H; ++y)
                                for (int x = x0; x < x0 + 16 && x < W; ++x) {
                                    const int yy = y + t / 3 - 1, xx = x + t % 3 - 1;
                                    const int ok = yy >= 0 && yy < H && xx >= 0 && xx < W;
                                    const float v = ok ? in[(((int64_t)n * CI + ci) * H + yy) * W + xx] : 0.0f;
                                    s = fmaf(g[(((int64_t)n * CO + co) * H + y) * W + x], v, s);
                                }
                        sum += s;
                    }
                dw[((int64_t)co * CI + ci) * 9 + t] = sum;
            }
}
