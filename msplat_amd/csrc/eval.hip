// eval.hip — the two image steps either side of a render: the RGBA8 display
// conversion and the evaluation metrics (PSNR, L1, SSIM) of a render against
// its target.
//
// RGBA8: Trainer::renderFromPoseToBuffer (msplat_api.mm:230-238) converts on
// the CPU: each channel min(max(v, 0), 1) * 255 truncated to a byte, alpha
// 255.  Here one thread per pixel writes its four bytes as one 32-bit store,
// so only 4 bytes per pixel cross to the host instead of 12.
//
// Metrics: psnr / l1_loss (model.cpp:25-40) and ssim_eval (ssim.cpp:61-123).
// SSIM blurs five maps per channel (x, y, x^2, y^2, xy) with a separable
// window_size-tap Gaussian whose borders clamp to the edge pixel
// (gaussianBlur, ssim.cpp:26-59), then averages
//   (2 mu_x mu_y + C1)(2 s_xy + C2) / ((mu_x^2 + mu_y^2 + C1)(s_x^2 + s_y^2 + C2))
// over pixels and channels, C1 = 0.01^2, C2 = 0.03^2.  One 256-thread
// workgroup per 64x16 output tile stages the tile plus a 5-pixel clamped
// halo of both images, one channel at a time, in LDS, takes the horizontal
// sums into LDS and the vertical sums from there.  Every per-pixel float is
// formed with the reference's operations in its order (horizontal pass
// first, taps summed from the first, products rounded before weighting), so
// per-pixel SSIM terms equal the CPU's; the sums over pixels are fp64 like
// the reference's, folded per workgroup and then over workgroups in a fixed
// order.
#include "common.hpp"
#include "kernels.hpp"

namespace msp {

namespace {

__global__ __launch_bounds__(256) void k_to_rgba8(const float* __restrict__ img, int64_t n,
                                                  uint32_t* __restrict__ rgba) {
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    uint32_t word = 0xFF000000u;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float v = fminf(fmaxf(img[3 * p + c], 0.f), 1.f) * 255.f;
        word |= (uint32_t)(uint8_t)v << (8 * c);
    }
    rgba[p] = word;
}

constexpr int EV_R = 5;                  // largest window radius (11 taps)
constexpr int EV_TW = 64, EV_TH = 16;    // output tile
constexpr int EV_IW = EV_TW + 2 * EV_R, EV_IH = EV_TH + 2 * EV_R;

// Sums of three doubles over the 256 threads of a block, fixed order; thread 0
// gets them (sh: 12 doubles).
__device__ __forceinline__ void block_sum3_f64(double (&v)[3], double* sh) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        for (int off = 32; off >= 1; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
        if ((threadIdx.x & 63) == 0) sh[4 * k + (threadIdx.x >> 6)] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] = (sh[4 * k] + sh[4 * k + 1]) + (sh[4 * k + 2] + sh[4 * k + 3]);
}

// Bound by instruction issue (11 taps of five sums, each a rounded product and
// an add, in both directions, without fused multiply-adds) and the latency
// around the barriers.  So a thread takes four neighbouring outputs: across,
// from one run of inputs read as float4 and with each product formed once;
// down, from one column of sums.  The pixels of all three channels are loaded
// at the start, 12 bytes a lane, and wait in registers for their turn in LDS.
// The window size is a template argument, so that the runs unroll.  1297x840:
// 46 us (one output a thread and a loop over the taps: 83 us).
template <int WS>
__global__ __launch_bounds__(256) void k_eval_tiles(const float* __restrict__ img,
                                                    const float* __restrict__ gt, int W, int H,
                                                    EvalWindow win, double* __restrict__ part) {
    constexpr int PAD = WS / 2, OFF = EV_R - PAD;   // taps k = 0..WS-1 read offsets k - PAD
    constexpr int PITCH = EV_IW + 2;                // float4 rows; the last run reads 2 past
    constexpr int NS = (EV_IH * EV_IW + 255) / 256;
    static_assert(EV_TW + 12 == PITCH && EV_TH == 16, "four rows of outputs per wave");
    __shared__ __align__(16) float s_r[EV_IH][PITCH];
    __shared__ __align__(16) float s_g[EV_IH][PITCH];
    __shared__ __align__(16) float s_h[5][EV_IH][EV_TW];
    __shared__ double s_red[12];
    const int x0 = blockIdx.x * EV_TW, y0 = blockIdx.y * EV_TH;
    const int tid = threadIdx.x;
    const float C1 = 0.01f * 0.01f, C2 = 0.03f * 0.03f;
    float pr[NS][3], pg[NS][3];
#pragma unroll
    for (int u = 0; u < NS; ++u) {
        const int i = min(tid + 256 * u, EV_IH * EV_IW - 1);
        const int r = i / EV_IW, col = i - r * EV_IW;
        const int sy = min(max(y0 - EV_R + r, 0), H - 1);
        const int sx = min(max(x0 - EV_R + col, 0), W - 1);
        const size_t s = 3 * ((size_t)sy * W + sx);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            pr[u][c] = img[s + c];
            pg[u][c] = gt[s + c];
        }
    }
    double sum[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (c) __syncthreads();
#pragma unroll
        for (int u = 0; u < NS; ++u) {
            const int i = tid + 256 * u, r = i / EV_IW, col = i - r * EV_IW;
            if (i < EV_IH * EV_IW) {
                s_r[r][col] = pr[u][c];
                s_g[r][col] = pg[u][c];
            }
        }
        __syncthreads();
        // rows the window's taps reach
        for (int i = tid; i < (EV_TH + WS - 1) * (EV_TW / 4); i += 256) {
            const int r = OFF + i / (EV_TW / 4), g = 4 * (i % (EV_TW / 4));
            float x[16], y[16];
#pragma unroll
            for (int j = 0; j < 16; j += 4) {
                const float4 a = *reinterpret_cast<const float4*>(&s_r[r][g + j]);
                const float4 b = *reinterpret_cast<const float4*>(&s_g[r][g + j]);
                x[j] = a.x; x[j + 1] = a.y; x[j + 2] = a.z; x[j + 3] = a.w;
                y[j] = b.x; y[j + 1] = b.y; y[j + 2] = b.z; y[j + 3] = b.w;
            }
            float a[5][4] = {};
#pragma unroll
            for (int j = OFF; j < OFF + WS + 3; ++j) {
                const float v[5] = {x[j], y[j], x[j] * x[j], y[j] * y[j], x[j] * y[j]};
#pragma unroll
                for (int o = 0; o < 4; ++o) {
                    const int k = j - OFF - o;
                    if (k < 0 || k >= WS) continue;
#pragma unroll
                    for (int m = 0; m < 5; ++m) a[m][o] += v[m] * win.w[k];
                }
            }
#pragma unroll
            for (int m = 0; m < 5; ++m)
                *reinterpret_cast<float4*>(&s_h[m][r][g]) = make_float4(a[m][0], a[m][1], a[m][2], a[m][3]);
        }
        __syncthreads();
        const int ox = tid & 63, oy = 4 * (tid >> 6);
        float a[5][4] = {};
#pragma unroll
        for (int j = 0; j < WS + 3; ++j) {
#pragma unroll
            for (int m = 0; m < 5; ++m) {
                const float v = s_h[m][oy + OFF + j][ox];
#pragma unroll
                for (int o = 0; o < 4; ++o) {
                    const int k = j - o;
                    if (k >= 0 && k < WS) a[m][o] += v * win.w[k];
                }
            }
        }
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            if (y0 + oy + o >= H || x0 + ox >= W) continue;
            const float mu1 = a[0][o], mu2 = a[1][o];
            const float m1sq = mu1 * mu1, m2sq = mu2 * mu2, m12 = mu1 * mu2;
            const float sig1sq = a[2][o] - m1sq, sig2sq = a[3][o] - m2sq, sig12 = a[4][o] - m12;
            const float num = (2.0f * m12 + C1) * (2.0f * sig12 + C2);
            const float den = (m1sq + m2sq + C1) * (sig1sq + sig2sq + C2);
            sum[0] += (double)(num / den);
            const float d = s_r[oy + o + EV_R][ox + EV_R] - s_g[oy + o + EV_R][ox + EV_R];
            sum[1] += (double)d * (double)d;
            sum[2] += (double)fabsf(d);
        }
    }
    const size_t b = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
    block_sum3_f64(sum, s_red);
    if (tid < 3) part[3 * b + tid] = tid == 0 ? sum[0] : tid == 1 ? sum[1] : sum[2];
}

// Sum of the nb workgroup partials (3 each), fixed order, into out[3].
__global__ __launch_bounds__(256) void k_eval_fold(const double* __restrict__ part, int nb,
                                                   double* __restrict__ out) {
    __shared__ double s_red[12];
    double v[3] = {0.0, 0.0, 0.0};
    for (int b = threadIdx.x; b < nb; b += 256)
#pragma unroll
        for (int k = 0; k < 3; ++k) v[k] += part[3 * (size_t)b + k];
    block_sum3_f64(v, s_red);
    if (threadIdx.x < 3) out[threadIdx.x] = threadIdx.x == 0 ? v[0] : threadIdx.x == 1 ? v[1] : v[2];
}

}  // namespace

int64_t eval_partial_count(int H, int W) {
    return (int64_t)((W + EV_TW - 1) / EV_TW) * ((H + EV_TH - 1) / EV_TH);
}

void launch_to_rgba8(hipStream_t s, const float* img, int64_t n, uint32_t* rgba) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_to_rgba8, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, img, n,
                       rgba);
}

void launch_image_metrics(hipStream_t s, const float* img, const float* gt, int H, int W,
                          const EvalWindow& win, double* part, double* out3) {
    const dim3 grid((W + EV_TW - 1) / EV_TW, (H + EV_TH - 1) / EV_TH);
    decltype(&k_eval_tiles<11>) tiles = win.ws == 1   ? k_eval_tiles<1>
                                        : win.ws == 3 ? k_eval_tiles<3>
                                        : win.ws == 5 ? k_eval_tiles<5>
                                        : win.ws == 7 ? k_eval_tiles<7>
                                        : win.ws == 9 ? k_eval_tiles<9>
                                                      : k_eval_tiles<11>;
    hipLaunchKernelGGL(tiles, grid, dim3(256), 0, s, img, gt, W, H, win, part);
    hipLaunchKernelGGL(k_eval_fold, dim3(1), dim3(256), 0, s, (const double*)part,
                       (int)(grid.x * grid.y), out3);
}

}  // namespace msp
