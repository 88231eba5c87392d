// ssim.hip — separable 11-tap SSIM + L1 loss, forward and backward, in one
// LDS-staged tile kernel.
//
// The reference's training semantics, in five separable passes per channel:
//   h-fwd        ssim_h_fwd_kernel (.metal:3053-3115): horizontal
//                zero-padded sums of x = gt, y = render (mu_x, mu_y, E[x^2],
//                E[y^2], E[xy]) at the in-image positions
//   v-fwd + h-bwd  ssim_fused_v_fwd_h_bwd_kernel (.metal:3226-3313): the
//                vertical sums -> SSIM and its derivative fields f1, f2, f3
//                at every centre of the in-image rows, including the 5-column
//                halo outside the image (whose zero statistics give
//                f = (0, -2/C2, 2/C2)), then the mirrored horizontal pass
//   v-bwd        ssim_v_bwd_kernel (.metal:3396-3464): mirrored vertical pass
//                (rows outside the image contribute nothing) and the
//                combination with the L1 sign term.
// One workgroup computes all five for a TX x TY block of output pixels,
// recomputing the halo each pass needs (rows +-10, columns +-10 of input)
// instead of passing the horizontal-backward fields through memory: the
// only HBM traffic is the two images with their halo and the gradient image.
// Every sum is accumulated in the same order as the reference's separate
// kernels, so the fusion changes no bit of the gradient image.  Each window
// term is added with one fused multiply-add (w gv gv as the product w gv,
// then an fma with gv): the reference writes a product and a sum, which its
// fast-math Metal build may contract the same way; the CPU oracle evaluates
// exactly these operations.
// The loss is reduced per workgroup into (sum SSIM, sum L1, pixel count) and
// folded in a fixed order by one workgroup of the next kernel (loss_fold in
// kernels.hpp); it equals the sum over pixels of
// w*(1 - mean_c SSIM) + (1-w)*mean_c |gt - r|.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace msp {

namespace {

constexpr int HALF = 5;
constexpr int WIN = 11;

// Tile of TX x TY output pixels, NT threads, and the regions of its passes
// (rows / columns relative to the tile's first output pixel (x0, y0)):
//   input (gt, render)    rows -10 .. TY+9,  columns -10 .. TX+9   IN_H x IN_W
//   horizontal sums       rows -10 .. TY+9,  columns -5 .. TX+4    IN_H x FD_W
//   fields f1, f2, f3     rows -5 .. TY+4,   columns -5 .. TX+4    FD_H x FD_W
//   horizontal backward   rows -5 .. TY+4,   columns 0 .. TX-1     FD_H x TX
//   vertical backward     rows 0 .. TY-1,    columns 0 .. TX-1     the outputs
// For 32 x 32 outputs the horizontal sums are evaluated 2.13 times per
// output, the fields 1.72 times and the horizontal backward 1.31 times (16 x
// 16: 3.66, 2.64 and 1.63 times).
// Bound by vector issue, LDS reads and the latency between barriers, so every
// pass's item takes a run of neighbouring positions: KH of a row for the
// horizontal sums, KV of a column for the vertical ones, KB of a row and KO of
// a column for the backward passes.  A run's inputs (ten more than its
// positions) are read once, where one position an item reads eleven each, and
// its positions are independent chains of multiply-adds.
// LDS layouts (64 banks of 4 bytes; 16-byte reads are served 16 lanes at a
// time): in the two horizontal passes consecutive lanes take consecutive rows,
// whose strides are odd numbers of 16-byte groups, and in the two vertical
// ones consecutive columns, so that neither reads nor writes share banks
// (but where a wave wraps from one run to the next).
//  * input: (gt, render) of a position as one float2, read two at a time
//  * horizontal sums: (mu_x, mu_y, E[x^2], E[y^2]) as a float4 and E[xy] as a float
//  * fields (f1, f2, f3) and horizontal backward (h1, h2, h3) as a float4 each
// The input and the fields share one LDS area, the horizontal sums and the
// horizontal backward another (each pass reads one and writes the other).
template <int TX_, int TY_, int NT_, int KH_, int KV_, int KB_, int KO_, int WAVES_>
struct Tile {
    static constexpr int TX = TX_, TY = TY_, NT = NT_, KH = KH_, KV = KV_, KB = KB_, KO = KO_;
    static constexpr int WAVES = WAVES_;                                   // per SIMD
    static constexpr int IN_W = TX + 4 * HALF, IN_H = TY + 4 * HALF;
    static constexpr int FD_W = TX + 2 * HALF, FD_H = TY + 2 * HALF;
    static constexpr int NH = (FD_W + KH - 1) / KH, NV = (FD_H + KV - 1) / KV;   // runs
    static constexpr int odd(int v) { return v | 1; }
    static constexpr int IN_S = 2 * odd((NH * KH + 2 * HALF + 1) / 2);      // row strides
    static constexpr int HS_S = odd(FD_W), FD_S = odd(FD_W), HB_S = odd(TX);
    static constexpr int HS_H = NV * KV + 2 * HALF;                         // rows the runs read
    static constexpr int cmax(int a, int b) { return a > b ? a : b; }
    static constexpr int LDS_A = cmax(IN_H * IN_S * 8, FD_H * FD_S * 16);
    static constexpr int LDS_B = cmax(HS_H * HS_S * (16 + 4), FD_H * HB_S * 16);
    static constexpr int NPOS = (IN_H * IN_W + NT - 1) / NT;                // input positions per thread
    static_assert(KH % 2 == 0 && TX % KB == 0 && TY % KO == 0, "runs");
    static_assert(TX * TY / KO <= NT, "one run of outputs per thread");
};

template <class G>
__global__ __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(G::WAVES))) void k_ssim_tile(
    int W, int H, const float* __restrict__ img, const float* __restrict__ gt, float w_ssim,
    float inv_n, float* __restrict__ v_rendered, float* __restrict__ loss_part) {
    constexpr int TX = G::TX, TY = G::TY, NT = G::NT, KH = G::KH, KV = G::KV, KB = G::KB, KO = G::KO;
    constexpr int IN_W = G::IN_W, IN_H = G::IN_H, FD_W = G::FD_W, FD_H = G::FD_H, NPOS = G::NPOS;
    constexpr int IN_S = G::IN_S, HS_S = G::HS_S, FD_S = G::FD_S, HB_S = G::HB_S;
    __shared__ __align__(16) char lds_a[G::LDS_A];
    __shared__ __align__(16) char lds_b[G::LDS_B];
    __shared__ float s_red[3][NT / 64];
    float2* s_in = reinterpret_cast<float2*>(lds_a);
    float4* s_f = reinterpret_cast<float4*>(lds_a);
    float4* s_h4 = reinterpret_cast<float4*>(lds_b);
    float* s_h1 = reinterpret_cast<float*>(lds_b + G::HS_H * HS_S * 16);
    float4* s_hb = reinterpret_cast<float4*>(lds_b);
    const int t = threadIdx.x;
    const int x0 = blockIdx.x * TX, y0 = blockIdx.y * TY;
    float ssim_sum = 0.f, l1_sum = 0.f, cnt = 0.f;
    // The three channels of this thread's input positions (zero outside the
    // image) are loaded once, into registers; each channel pass copies its
    // component into LDS.
    float rg[NPOS][3], rr[NPOS][3];
#pragma unroll
    for (int k = 0; k < NPOS; ++k) {
        const int i = t + k * NT;
        const int iy = i / IN_W, ix = i - iy * IN_W;
        const int gy = y0 - 2 * HALF + iy, gx = x0 - 2 * HALF + ix;
        const bool in = i < IN_H * IN_W && gx >= 0 && gx < W && gy >= 0 && gy < H;
        const size_t q = in ? ((size_t)gy * W + gx) * 3 : 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            rg[k][c] = gt[q + c];
            rr[k][c] = img[q + c];
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            rg[k][c] = in ? rg[k][c] : 0.f;
            rr[k][c] = in ? rr[k][c] : 0.f;
        }
    }
    // this thread's output pixels: column ox, rows oy .. oy + KO - 1
    const int ox = t % TX, oy = (t / TX) * KO;
    const int gox = x0 + ox, goy = y0 + oy;
    const int n_out = oy < TY && gox < W ? min(KO, H - goy) : 0;   // may be negative
    float vr[KO][3] = {};
#pragma unroll
    for (int u = 0; u < KO; ++u) cnt += u < n_out ? 1.f : 0.f;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        // the previous channel's vertical backward has read the horizontal
        // backward before this channel's sums overwrite it, and its fields
        // are consumed
        if (c > 0) __syncthreads();
#pragma unroll
        for (int k = 0; k < NPOS; ++k) {
            const int i = t + k * NT;
            if (i < IN_H * IN_W) {
                const int iy = i / IN_W, ix = i - iy * IN_W;
                s_in[iy * IN_S + ix] = make_float2(rg[k][c], rr[k][c]);
            }
        }
        __syncthreads();
        // horizontal zero-padded sums (ssim_h_fwd, .metal:3094-3114) at the
        // in-image positions; zero elsewhere.  Input k of a run is term k - u
        // of the sums of its position u, each added in the reference's order.
        // (A last run may read past the input's columns, for positions past
        // FD_W that it does not store.)
        for (int i = t; i < IN_H * G::NH; i += NT) {
            const int hg = i / IN_H, hy = i - hg * IN_H, hx = KH * hg;
            const int gy = y0 - 2 * HALF + hy, gx = x0 - HALF + hx;
            const bool rin = gy >= 0 && gy < H;
            float acc[KH][5] = {};
            const float4* row = reinterpret_cast<const float4*>(s_in + hy * IN_S + hx);
#pragma unroll
            for (int q = 0; q < (KH + WIN - 1) / 2; ++q) {
                const float4 f = row[q];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int k = 2 * q + e;
                    const float gv = e ? f.z : f.x, rv = e ? f.w : f.y;
#pragma unroll
                    for (int u = 0; u < KH; ++u) {
                        const int d = k - u;
                        if (d < 0 || d >= WIN) continue;
                        const float w = GAUSS_1D[d];
                        const float wg = w * gv, wr = w * rv;
                        acc[u][0] = fmaf(w, gv, acc[u][0]);
                        acc[u][1] = fmaf(w, rv, acc[u][1]);
                        acc[u][2] = fmaf(wg, gv, acc[u][2]);
                        acc[u][3] = fmaf(wr, rv, acc[u][3]);
                        acc[u][4] = fmaf(wg, rv, acc[u][4]);
                    }
                }
            }
            const int o = hy * HS_S + hx;
#pragma unroll
            for (int u = 0; u < KH; ++u) {
                const bool in = rin && gx + u >= 0 && gx + u < W;
                if (FD_W % KH != 0 && hx + u >= FD_W) continue;
                s_h4[o + u] = make_float4(in ? acc[u][0] : 0.f, in ? acc[u][1] : 0.f, in ? acc[u][2] : 0.f,
                                          in ? acc[u][3] : 0.f);
                s_h1[o + u] = in ? acc[u][4] : 0.f;
            }
        }
        __syncthreads();
        // vertical sums, SSIM and the derivative fields (.metal:3243-3300)
        // at the centres of the in-image rows (the fields of other rows are
        // never read: their horizontal backward is zero).  Row k of a run is
        // term k - u of the sums of its row u, each added in order.
        for (int i = t; i < G::NV * FD_W; i += NT) {
            const int fy0 = KV * (i / FD_W), fx = i - (i / FD_W) * FD_W;
            const int gx = x0 - HALF + fx;
            float acc[KV][5] = {};
#pragma unroll
            for (int k = 0; k < KV + WIN - 1; ++k) {
                const float4 q = s_h4[(fy0 + k) * HS_S + fx];
                const float q4 = s_h1[(fy0 + k) * HS_S + fx];
#pragma unroll
                for (int u = 0; u < KV; ++u) {
                    const int d = k - u;
                    if (d < 0 || d >= WIN) continue;
                    const float w = GAUSS_1D[d];
                    acc[u][0] = fmaf(w, q.x, acc[u][0]);
                    acc[u][1] = fmaf(w, q.y, acc[u][1]);
                    acc[u][2] = fmaf(w, q.z, acc[u][2]);
                    acc[u][3] = fmaf(w, q.w, acc[u][3]);
                    acc[u][4] = fmaf(w, q4, acc[u][4]);
                    // the sums are formed row by row (without this the compiler
                    // sinks them into the per-row validity test and keeps all
                    // rows in registers, which spills)
                    asm volatile("" : "+v"(acc[u][0]), "+v"(acc[u][1]), "+v"(acc[u][2]), "+v"(acc[u][3]),
                                 "+v"(acc[u][4]));
                }
            }
#pragma unroll
            for (int u = 0; u < KV; ++u) {
                const int fy = fy0 + u;
                const int gy = y0 - HALF + fy;
                if (gy < 0 || gy >= H || (FD_H % KV != 0 && fy >= FD_H)) continue;
                const float mx = acc[u][0], my = acc[u][1], sx = acc[u][2], sy = acc[u][3],
                            cxy = acc[u][4];
                const float sxs = sx - mx * mx, sys = sy - my * my, sxy = cxy - mx * my;
                const float A = 2.0f * mx * my + SSIM_C1, B = 2.0f * sxy + SSIM_C2;
                const float Cd = mx * mx + my * my + SSIM_C1, D = sxs + sys + SSIM_C2;
                const float iCD = 1.0f / (Cd * D);
                const float dmu = 2.0f * B * (mx * Cd - A * my) / (Cd * Cd * D);
                const float dsyq = -A * B * iCD / D, dsxy = 2.0f * A * iCD;
                s_f[fy * FD_S + fx] = make_float4(dmu - 2.0f * my * dsyq - mx * dsxy, 2.0f * dsyq, dsxy, 0.f);
                // the tile's own in-image outputs add their SSIM to the loss
                if (fy >= HALF && fy < HALF + TY && fx >= HALF && fx < HALF + TX && gx >= 0 && gx < W)
                    ssim_sum += (A * B) / (Cd * D);
            }
        }
        // this thread's output pixels of the channel, for the last pass
        float og[KO], orr[KO];
#pragma unroll
        for (int u = 0; u < KO; ++u) {
            const size_t q = u < n_out ? ((size_t)(goy + u) * W + gox) * 3 + c : 0;
            og[u] = gt[q];
            orr[u] = img[q];
        }
        __syncthreads();
        // mirrored horizontal backward at the in-image rows of the tile's
        // columns +- 5 rows (zero at rows outside the image, whose fields are
        // not formed)
        for (int i = t; i < FD_H * (TX / KB); i += NT) {
            const int bg = i / FD_H, by = i - bg * FD_H, bx = KB * bg;
            const int gy = y0 - HALF + by;
            float h[KB][3] = {};
            if (gy >= 0 && gy < H) {
                const float4* fr = s_f + by * FD_S + bx;
#pragma unroll
                for (int k = 0; k < KB + WIN - 1; ++k) {
                    const float4 f = fr[k];
#pragma unroll
                    for (int u = 0; u < KB; ++u) {
                        const int d = k - u;
                        if (d < 0 || d >= WIN) continue;
                        const float w = GAUSS_1D[WIN - 1 - d];
                        h[u][0] = fmaf(w, f.x, h[u][0]);
                        h[u][1] = fmaf(w, f.y, h[u][1]);
                        h[u][2] = fmaf(w, f.z, h[u][2]);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < KB; ++u) s_hb[by * HB_S + bx + u] = make_float4(h[u][0], h[u][1], h[u][2], 0.f);
        }
        __syncthreads();
        // mirrored vertical backward (.metal:3443-3463) and the L1 term
        if (n_out > 0) {
            float f[KO][3] = {};
            const float4* hr = s_hb + oy * HB_S + ox;
#pragma unroll
            for (int k = 0; k < KO + WIN - 1; ++k) {
                const float4 h = hr[k * HB_S];
#pragma unroll
                for (int u = 0; u < KO; ++u) {
                    const int d = k - u;
                    if (d < 0 || d >= WIN) continue;
                    const float w = GAUSS_1D[WIN - 1 - d];
                    f[u][0] = fmaf(w, h.x, f[u][0]);
                    f[u][1] = fmaf(w, h.y, f[u][1]);
                    f[u][2] = fmaf(w, h.z, f[u][2]);
                }
            }
#pragma unroll
            for (int u = 0; u < KO; ++u) {
                const float r = orr[u], g = og[u];
                const float v_ssim = f[u][0] + r * f[u][1] + g * f[u][2];
                const float v_l1 = (g > r) ? -1.0f : ((g < r) ? 1.0f : 0.0f);
                vr[u][c] = inv_n * (-w_ssim * v_ssim + (1.0f - w_ssim) * v_l1);
                l1_sum += u < n_out ? fabsf(g - r) : 0.f;
            }
        }
    }
#pragma unroll
    for (int u = 0; u < KO; ++u) {
        if (u >= n_out) continue;
        const size_t q = ((size_t)(goy + u) * W + gox) * 3;
        v_rendered[q + 0] = vr[u][0];
        v_rendered[q + 1] = vr[u][1];
        v_rendered[q + 2] = vr[u][2];
    }
    // Workgroup partials of (sum SSIM, sum L1, pixels).
    const float a = wave_sum(ssim_sum), b = wave_sum(l1_sum), n = wave_sum(cnt);
    if ((t & 63) == 0) {
        s_red[0][t >> 6] = a;
        s_red[1][t >> 6] = b;
        s_red[2][t >> 6] = n;
    }
    __syncthreads();
    if (t < 3) {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < NT / 64; ++k) v += s_red[t][k];
        loss_part[((size_t)blockIdx.y * gridDim.x + blockIdx.x) * 3 + t] = v;
    }
}

// The tile by the size of the image.  A call takes about as long as its
// rounds of workgroups: 256 CUs hold two of the larger tiles each.
//  * 16 x 16 while every tile gets a CU of its own: the chain of passes is
//    shortest (256x256: 11.1 us, against 15.0 with 32 x 24 and 18.0 with 32 x 32)
//  * else 32 x 32, which recomputes the least halo, or 32 x 24, whose round
//    takes 5/6 of the time, whichever makes less of the rounds (1297x840: 61.2
//    us in three rounds against 64.7 in three; 2594x1680: 204 us in nine against
//    220 in twelve; 800x600: 28.4 us in one against 33.2 in two)
// One pass position per item and 32 x 32 tiles for all took 19.3 us at
// 256x256, 30.3 at 648x420, 67.8 at 1297x840 and 217 at 2594x1680.
using TileS = Tile<16, 16, 512, 2, 2, 1, 1, 8>;
using TileM = Tile<32, 24, 512, 4, 3, 4, 2, 4>;
using TileL = Tile<32, 32, 512, 6, 4, 4, 2, 4>;
constexpr int CUS = 256;

template <class G>
int tiles(int W, int H) {
    return ((W + G::TX - 1) / G::TX) * ((H + G::TY - 1) / G::TY);
}

template <class G>
int run(hipStream_t s, int H, int W, const float* img, const float* gt, float w, float inv_n,
        float* v_rendered, float* loss_part) {
    const dim3 grid((W + G::TX - 1) / G::TX, (H + G::TY - 1) / G::TY);
    hipLaunchKernelGGL(k_ssim_tile<G>, grid, dim3(G::NT), 0, s, W, H, img, gt, w, inv_n, v_rendered,
                       loss_part);
    return tiles<G>(W, H);
}

}  // namespace

int ssim_part_bound(int H, int W) {
    return std::max({tiles<TileS>(W, H), tiles<TileM>(W, H), tiles<TileL>(W, H)});
}

int launch_ssim(hipStream_t s, int H, int W, const float* img, const float* gt, float w,
                float inv_n, float* v_rendered, float* loss_part) {
    const auto rounds = [](int n) { return (n + 2 * CUS - 1) / (2 * CUS); };
    if (tiles<TileS>(W, H) <= CUS) return run<TileS>(s, H, W, img, gt, w, inv_n, v_rendered, loss_part);
    if (5 * rounds(tiles<TileM>(W, H)) < 6 * rounds(tiles<TileL>(W, H)))
        return run<TileM>(s, H, W, img, gt, w, inv_n, v_rendered, loss_part);
    return run<TileL>(s, H, W, img, gt, w, inv_n, v_rendered, loss_part);
}

}  // namespace msp
