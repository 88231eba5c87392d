// raster.hip — alpha compositing forward, chunk merge and backward.
//
// Work decomposition: one 256-thread workgroup (four wave64) per (tile,
// chunk) item; each wave owns one 8x8 quadrant of the 16x16 tile and each of
// its 16-lane rows one 4x4 block of that quadrant, one lane per pixel.
// Sorted entries (gaussian ids; each entry's projection record is gathered by
// id) are staged through LDS 256 at a time; every row walks the list of the
// staged entries that reach its block.  A tile that is rasterised in one piece writes the
// final image directly; a chunked tile writes per-pixel chunk state that the
// merge kernel folds front to back.
//
// Semantics follow the reference exactly:
//   forward      nd_rasterize_forward_kernel (.metal:472-585)
//   chunked fwd  rasterize_forward_chunked_kernel (.metal:2633-2741)
//   merge        rasterize_forward_merge_kernel (.metal:2746-2799)
//   prefix/sfx   compute_chunk_prefix_suffix_kernel (.metal:2804-2840)
//   backward     rasterize_backward_kernel (.metal:898-1099) and
//                rasterize_backward_chunked_kernel (.metal:2844-3031)
// with these MI355X differences: each loaded entry carries a conservative
// mask of the tile's sixteen 4x4 blocks it can reach and a row of lanes walks
// only the entries of its own block; a workgroup-wide vote stops the forward once
// every pixel of the item has terminated; the backward holds 16 entries in a
// row's lanes, scans what a pixel carries from one to the next, and adds a
// window's gradient sums to memory with consecutive lanes on consecutive floats.
#include "common.hpp"
#include "kernels.hpp"

#include <utility>

namespace msp {

namespace {

struct Px {
    int i, j;      // pixel row / column
    int lp;        // local pixel index within the tile (ly * 16 + lx)
    bool inside;
};

// Pixel of thread tid of the tile's 256.
__device__ __forceinline__ Px pixel_at(int t, int tbx, int W, int H, int tid) {
    const int w = tid >> 6, r = (tid >> 4) & 3, i = tid & 15;
    const int lx = (w & 1) * 8 + (r & 1) * 4 + (i & 3), ly = (w >> 1) * 8 + (r >> 1) * 4 + (i >> 2);
    Px p;
    p.j = (t % tbx) * BLOCK + lx;
    p.i = (t / tbx) * BLOCK + ly;
    p.lp = ly * BLOCK + lx;
    p.inside = p.i < H && p.j < W;
    return p;
}
__device__ __forceinline__ Px pixel_of(int t, int tbx, int W, int H) {
    return pixel_at(t, tbx, W, H, threadIdx.x);
}

// Lanes below this one in a lane mask.
__device__ __forceinline__ int lanes_below(uint64_t m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Pair counters: WORK_SLOTS copies of the counter set, one 128-byte line
// each, picked by block id, so that the atomics of concurrent workgroups do
// not serialise on one address; the host sums the slots.
__device__ __forceinline__ unsigned long long* work_slot(unsigned long long* work) {
    return work + (size_t)(blockIdx.x % WORK_SLOTS) * WORK_SLOT_U64;
}

// Conservative block mask of one entry: bit 4 w + r is set when the entry can
// reach alpha >= 1/255 at a pixel of the 4x4 block of row r of wave w, in the
// tile at (tx0, ty0).  The reach is the ellipse sigma < min(5.55, ln(255 o)),
// with margins on that threshold and of 1/32 pixel around the blocks.  For the
// tile's four strips of 4 pixel rows, the part of the ellipse inside a strip
// spans an interval of x whose ends are the ellipse's extremes with their
// offset dy clamped to the strip (the ellipse is convex); the blocks of the
// strip that meet the interval are set.  Entries outside a block are ones the
// per-pixel tests skip there, so culling them changes no result.
// The threshold's margin covers what a pixel's computed sigma may be below its
// value: the terms a dx^2, c dy^2 and b dx dy of a needle cancel, each up to 2
// kappa sigma with kappa = a c / (a c - b^2), and the roundings that fwd_step
// makes on them add up to at most 17 u kappa sigma (u = 2^-24; the bound is
// taken 1.08 times).  Where that is half of sigma (needles of 1000 pixels and
// more), nothing is culled.  About 140 vector instructions (the four exact
// quadrant minima that a coarser mask of 8x8 quadrants took were 250).
__device__ __forceinline__ int block_mask(float x, float y, float a, float b, float c, float o,
                                          int tx0, int ty0) {
    if (!(o >= 0.0039f)) return o == o ? 0 : 0xFFFF;   // alpha <= o < 1/255 everywhere
    // a c - b^2 with the rounding error of b^2 put back: needle-shaped conics
    // leave few bits of the plain difference
    const float bb = b * b;
    const float det = fmaf(a, c, -bb) - fmaf(b, b, -bb);
    if (!(det > 1e-30f) || !(det < 1e30f) || !(a > 0.f) || !(c > 0.f) || !(a < 1e30f) ||
        !(c < 1e30f) || !(fabsf(x) < 1e30f) || !(fabsf(y) < 1e30f))
        return 0xFFFF;
    constexpr float M = 0.03125f;
    const float ia = __builtin_amdgcn_rcpf(a), id = __builtin_amdgcn_rcpf(det);
    const float err = 1.1e-6f * (a * c * id);     // of sigma, relative
    if (!(err < 0.5f)) return 0xFFFF;
    // sigma (1 - err) <= t holds up to sigma = t / (1 - err) <= t (1 + 2 err)
    const float thr2 = 2.f * (fminf(5.55f, __logf(255.f * o) + 0.05f) * 1.002f + 1e-3f) * fmaf(2.f, err, 1.f);
    // offsets d = centre - pixel: at offset dy the ellipse spans dx = (-b dy
    // -+ sqrt(a thr2 - det dy^2)) / a; its largest dx lies at dy = -k
    const float k = b * __builtin_amdgcn_rcpf(c) * __builtin_amdgcn_sqrtf(c * thr2 * id);
    const float at = a * thr2, ymax = __builtin_amdgcn_sqrtf(at * id);
    const float cx = x - (float)tx0, cy = y - (float)ty0;
    int m = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float d0 = cy - (4 * q + 3 + M), d1 = cy - (4 * q - M);
        const float yl = __builtin_amdgcn_fmed3f(-k, d0, d1), yr = __builtin_amdgcn_fmed3f(k, d0, d1);
        const float el = fmaf(-det * yl, yl, at), er = fmaf(-det * yr, yr, at);
        // pixel interval [cx - largest dx, cx - smallest dx] in tile coordinates
        const float l = cx - fmaf(-b, yl, __builtin_amdgcn_sqrtf(fmaxf(el, 0.f))) * ia - M;
        const float r = cx - fmaf(-b, yr, -__builtin_amdgcn_sqrtf(fmaxf(er, 0.f))) * ia + M;
        const int j0 = (int)fminf(fmaxf(ceilf((l - 3.f) * 0.25f), 0.f), 4.f);
        const int j1 = (int)fminf(fmaxf(floorf(r * 0.25f), -1.f), 3.f);
        int s = (0xF << j0) & (0xF >> (3 - j1)) & 0xF;
        if (d0 > ymax || d1 < -ymax) s = 0;           // the strip misses the ellipse
        const int sh = 8 * (q >> 1) + 2 * (q & 1);
        m |= (s & 3) << sh | (s >> 2) << (sh + 4);
    }
    return m;
}

// The reference's range early-out, skip when sigma < 0 || sigma >= 5.55
// (.metal:551, 1029, 2718, 2976), folded into the alpha test: sigma's bits
// are clamped with one unsigned min to those of 5.55f (0x40B1999A), so sigma
// in [+0, 5.55) keeps its value and everything else (negative, -0, >= 5.55,
// +inf, NaN) becomes 5.55, where alpha = min(0.999, o exp(-5.55)) <=
// 0.0038875 < 1/255 for every opacity in [0, 1] and the alpha test rejects
// the pair.  One vector min replaces two compares and two scalar ands per
// entry step; the decision differs from the reference's only for sigma = -0
// or NaN (a degenerate conic), which are rejected here, and for a NaN
// opacity (alpha 0.999 wherever the entry is walked).
__device__ __forceinline__ float sigma_clamp(float s) {
    return __uint_as_float(min(__float_as_uint(s), 0x40B1999Au));
}

// Entry record at byte offset qb of an LDS array of float4.
__device__ __forceinline__ float4 lds_f4(const float4* base, int qb) {
    return *static_cast<const float4*>(
        __builtin_assume_aligned(reinterpret_cast<const char*>(base) + qb, 16));
}

// Byte offset of the dummy record behind the staged ones: opacity 0, no pixel
// takes it.
constexpr int DUMMY = 256;

// The value of lane N of each row of 16, in all lanes of the row.
template <int N>
__device__ __forceinline__ int row_bcast(int v) {
    return __builtin_amdgcn_mov_dpp(v, 0x150 + N, 0xF, 0xF, true);
}

// Entry lists of a wave's four rows: the batch's entries whose mask (s_mask,
// one per staged entry, bit 4 w + r) names the row's block, in order, as one
// byte each in s_list[256 r ...].  Returns this lane's
// row's count; longest is the largest of the four (both wave-uniform per row).
// Costs about 9 instructions per row and 64 entries.  Where at most 64 entries
// of the 256 reach the wave's quadrant (long lists of needles, whose rectangles
// cover tiles that they miss), these are put together first, so that the rows
// are gone through once instead of four times: renders of 100k needles of sd 110
// pixels at 1297x840 589 -> 571 us, of 300k at 2000x1300 1529 -> 1495 (with
// 8 x 8 quadrants 600 and 1457); others the same (500k: 233.9 and 233.9).
__device__ __forceinline__ int build_lists(int w, const uint16_t* s_mask, uint8_t* s_list,
                                           int& longest) {
    const int lane = threadIdx.x & 63;
    int n[4] = {0, 0, 0, 0};
    unsigned m[4];
    int total = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        m[c] = ((unsigned)s_mask[64 * c + lane] >> (4 * w)) & 15u;
        total += __popcll(wave_ballot(m[c] != 0u));
    }
    auto rows = [&](int q, unsigned mq) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint64_t in = wave_ballot((mq >> r) & 1u);
            const int at = n[r] + lanes_below(in);
            if (lane_of(in)) s_list[256 * r + at] = (uint8_t)q;
            n[r] += __popcll(in);
        }
    };
    if (total <= 64) {
        // (entry, mask) pairs, behind the 64 places that a row can need
        uint16_t* pairs = reinterpret_cast<uint16_t*>(s_list + 128);
        int k = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint64_t in = wave_ballot(m[c] != 0u);
            if (lane_of(in)) pairs[k + lanes_below(in)] = (uint16_t)((64 * c + lane) << 4 | m[c]);
            k += __popcll(in);
        }
        __builtin_amdgcn_wave_barrier();
        const unsigned p = lane < total ? pairs[lane] : 0u;
        rows((int)(p >> 4), p & 15u);
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) rows(64 * c + lane, m[c]);
    }
    __builtin_amdgcn_wave_barrier();
    longest = max(max(n[0], n[1]), max(n[2], n[3]));
    const int row = lane >> 4;
    return row == 0 ? n[0] : row == 1 ? n[1] : row == 2 ? n[2] : n[3];
}

// LDS of a forward workgroup: 256 staged entries and the dummy.
struct FwdLds {
    float4 geo[257];         // x, y, conic a, b
    float4 col[257];         // conic c, opacity, clamped r, g
    float4 aux[257];         // clamped b; 16-byte stride shares the address
    uint16_t mask[256];      // block masks
    uint8_t list[4][4 * 256];   // per wave: its rows' entry lists
};

// One entry of the forward at this lane's pixel: qb is the byte offset of the
// entry's record, different from row to row.  A lane whose pixel has stopped
// (or lies outside the image) has thr = 2 and takes nothing.  Lanes without a
// hit run the same steps with alpha = 0, which leaves T and the colours as
// they are (the staged colours are finite); the rare step in which a pixel
// stops is put right in a branch.
template <bool COUNT>
__device__ __forceinline__ void fwd_step(int qb, float fx, float fy, const FwdLds& s, float& thr,
                                         float& T, float& C0, float& C1, float& C2, int& lqb,
                                         unsigned& ncl) {
    const float4 g = lds_f4(s.geo, qb);
    const float4 c = lds_f4(s.col, qb);
    const float cb = lds_f4(s.aux, qb).x;
    const float dx = g.x - fx, dy = g.y - fy;
    const float sigma = fmaf(0.5f, fmaf(g.z, dx * dx, c.x * dy * dy), g.w * dx * dy);
    const float alpha = fminf(0.999f, c.y * exp_neg_raster(sigma_clamp(sigma)));
    // hit: the pixel is live and alpha >= 1/255 (sigma out of range: alpha < 1/255)
    const bool hit = alpha >= thr;
    float a = hit ? alpha : 0.f;
    float nT = T * (1.f - a);
    lqb = hit ? qb : lqb;
    if (COUNT) ncl += hit ? 1u : 0u;
    // T > 1e-4 at every pixel, so only a hit can get here
    const uint64_t sm = mask_le(nT, 1e-4f);
    if (__builtin_expect(sm != 0, 0)) {      // once per pixel: this entry is not composited
        if (lane_of(sm)) {
            a = 0.f;
            nT = T;
            thr = 2.f;
            lqb = qb - (int)sizeof(float4);  // the entry before this one
            if (COUNT) --ncl;
        }
    }
    const float vis = a * T;
    C0 = fmaf(c.z, vis, C0);
    C1 = fmaf(c.w, vis, C1);
    C2 = fmaf(cb, vis, C2);
    T = nT;
}

// Four consecutive list entries (positions B .. B + 3 of the row's 16).
template <bool COUNT, int B>
__device__ __forceinline__ void fwd_four(int off, float fx, float fy, const FwdLds& s, float& thr,
                                         float& T, float& C0, float& C1, float& C2, int& lqb,
                                         unsigned& ncl) {
    fwd_step<COUNT>(row_bcast<B>(off), fx, fy, s, thr, T, C0, C1, C2, lqb, ncl);
    fwd_step<COUNT>(row_bcast<B + 1>(off), fx, fy, s, thr, T, C0, C1, C2, lqb, ncl);
    fwd_step<COUNT>(row_bcast<B + 2>(off), fx, fy, s, thr, T, C0, C1, C2, lqb, ncl);
    fwd_step<COUNT>(row_bcast<B + 3>(off), fx, fy, s, thr, T, C0, C1, C2, lqb, ncl);
}

// Colour of a staged entry's channel: clamped from below as the reference
// does, and finite, so that alpha = 0 composites nothing.
__device__ __forceinline__ float staged_colour(float raw) {
    return fminf(fmaxf(raw + 0.5f, 0.f), 3.402823466e38f);
}

// Bound: vector and scalar issue.  Rows with lists of their own take 2.23M wave
// steps where waves with one list for an 8 x 8 quadrant took 3.08M (1.5M
// gaussians at 1297x840), and a step has no scalar mask work: forward 165 ->
// 137 us there, 499 -> 402 us for a 1M blob at 2594x1680, 30 -> 20 us for 10k
// at 256x256, and in renders 118 -> 97 us (500k at 1297x840) and 1151 -> 1039
// us (6M at 4946x3286).
// Forward of the entries [cs, ce) at this lane's pixel, from the state
// (T, C, last) passed in: entries are staged 256 at a time through LDS and
// each row walks the entries of its block in order.  live: this lane's pixel
// still composites.  Every thread of the workgroup calls this with the same
// range (it holds workgroup barriers).
// MASKS (the training forward): each staged entry's block mask is also
// stored for the backward.
template <bool COUNT, bool MASKS = false>
__device__ __forceinline__ void fwd_range(int cs, int ce, bool live, float fx, float fy,
                                          int tx0, int ty0, const Entries& pk, FwdLds& s, float& T,
                                          float& C0, float& C1, float& C2, int& last,
                                          unsigned& ncl, unsigned& nwit) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    float thr = live ? 1.f / 255.f : 2.f;
    if (tid == 0) s.geo[DUMMY] = s.col[DUMMY] = s.aux[DUMMY] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int b = cs; b < ce; b += 256) {
        if (__syncthreads_and(thr > 1.f)) break;
        const int idx = b + tid;
        int mask = 0;
        if (idx < ce) {
            const float4* r = pk.rec + 4 * (size_t)pk.ids[idx];
            const float4 g = r[0];
            const float4 c = r[1];
            const float bl = r[2].x;
            mask = block_mask(g.x, g.y, g.z, g.w, c.x, c.y, tx0, ty0);
            if (MASKS) pk.bmask[idx] = (uint16_t)mask;
            s.geo[tid] = g;
            s.col[tid] = make_float4(c.x, c.y, staged_colour(c.z), staged_colour(c.w));
            s.aux[tid] = make_float4(staged_colour(bl), 0.f, 0.f, 0.f);
        }
        s.mask[tid] = (uint16_t)mask;
        __syncthreads();
        if (wave_ballot(thr < 1.f) == 0) continue;
        int longest;
        const int n = build_lists(w, s.mask, s.list[w], longest);
        const uint8_t* list = s.list[w] + 256 * (lane >> 4);
        // this batch's last contributor as the entry's LDS byte offset (a
        // vector register copy per step), turned into the index at the end
        int lqb = INT_MIN;
        for (int p = 0; p < longest; p += 16) {
            const int q = p + (lane & 15);
            const int off = (q < n ? (int)list[q] : DUMMY) * (int)sizeof(float4);
            if (COUNT) nwit += min(longest - p, 16);
            fwd_four<COUNT, 0>(off, fx, fy, s, thr, T, C0, C1, C2, lqb, ncl);
            if (p + 4 >= longest) break;
            fwd_four<COUNT, 4>(off, fx, fy, s, thr, T, C0, C1, C2, lqb, ncl);
            if (p + 8 >= longest) break;
            fwd_four<COUNT, 8>(off, fx, fy, s, thr, T, C0, C1, C2, lqb, ncl);
            if (p + 12 >= longest) break;
            fwd_four<COUNT, 12>(off, fx, fy, s, thr, T, C0, C1, C2, lqb, ncl);
            if (wave_ballot(thr < 1.f) == 0) break;
        }
        if (lqb != INT_MIN) last = b + (lqb >> 4);   // sizeof(float4) = 16; -16 gives b - 1
    }
}

template <bool COUNT>
__device__ __forceinline__ void add_work(unsigned long long* work, unsigned ncl, unsigned nwit) {
    if (!COUNT || !work) return;
    unsigned long long* ws = work_slot(work);
    unsigned ncomp = ncl;
    for (int off = 32; off >= 1; off >>= 1) ncomp += __shfl_xor(ncomp, off, 64);
    const int lane = threadIdx.x & 63;
    if (lane == 0 && ncomp) atomicAdd(ws, (unsigned long long)ncomp);
    if (lane == 0 && nwit) atomicAdd(ws + 2, (unsigned long long)nwit);
}

// One work item of the training forward: its chunk's state (chunked tile)
// or the tile's final pixels (tile in one piece).
template <bool COUNT>
__device__ __forceinline__ void fwd_item(int4 rec, int W, int H, int tbx, float bg0, float bg1,
                                         float bg2, const Entries& pk, float* final_T, int* final_idx,
                                         float* out_img, const ChunkBufs& cb,
                                         unsigned long long* work, FwdLds& s) {
    const int item = rec.x, t = rec.y & ITEM_TILE, cs = rec.z, ce = rec.w;
    const Px px = pixel_of(t, tbx, W, H);
    float fx = (float)px.j, fy = (float)px.i;
    // opaque to the compiler, so that the loop keeps the converted
    // coordinates instead of converting the integers again every step
    asm volatile("" : "+v"(fx), "+v"(fy));
    const int tx0 = (t % tbx) * BLOCK, ty0 = (t / tbx) * BLOCK;

    float T = 1.f, C0 = 0.f, C1 = 0.f, C2 = 0.f;
    int last = cs - 1;
    unsigned ncl = 0;       // pairs composited by this lane
    unsigned nwit = 0;      // entries this wave evaluated (wave-uniform)
    fwd_range<COUNT, true>(cs, ce, px.inside, fx, fy, tx0, ty0, pk, s, T, C0, C1, C2, last, ncl, nwit);
    add_work<COUNT>(work, ncl, nwit);
    if (!px.inside) return;
    if (!(rec.y & ITEM_MULTI)) {
        const size_t pix = (size_t)px.i * W + px.j;
        final_T[pix] = T;
        final_idx[pix] = last;
        out_img[3 * pix + 0] = clamp01(fmaf(bg0, T, C0));
        out_img[3 * pix + 1] = clamp01(fmaf(bg1, T, C1));
        out_img[3 * pix + 2] = clamp01(fmaf(bg2, T, C2));
    } else {
        const size_t o = (size_t)item * TILE_PIX + px.lp;
        cb.cT[o] = T;
        cb.cC[3 * o + 0] = C0;
        cb.cC[3 * o + 1] = C1;
        cb.cC[3 * o + 2] = C2;
        cb.cidx[o] = last;
    }
}

// Chunks 0 .. FWD_P - 1 of every tile, one item per workgroup.
template <bool COUNT>
__global__ __launch_bounds__(256) void k_raster_fwd(int W, int H, int tbx, float bg0, float bg1,
                                                    float bg2, const Meta* __restrict__ meta,
                                                    Items it, Entries pk,
                                                    float* __restrict__ final_T,
                                                    int* __restrict__ final_idx,
                                                    float* __restrict__ out_img, ChunkBufs cb,
                                                    unsigned long long* __restrict__ work) {
    __shared__ FwdLds s;
    // items in launch order (heaviest size class first)
    if ((int)blockIdx.x >= meta->n_items) return;
    const int4 rec = it.rec[blockIdx.x];
    if (rec.y & ITEM_LATE) return;
    fwd_item<COUNT>(rec, W, H, tbx, bg0, bg1, bg2, pk, final_T, final_idx, out_img, cb,
             work, s);
}

// Chunks FWD_P and later of the tiles not marked done: few items qualify, so a
// small grid visits them all, each thread looking at one item of its
// workgroup's next 256 and the workgroup rasterising those found.
template <bool COUNT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_raster_fwd_tail(int W, int H, int tbx,
                                                         const Meta* __restrict__ meta, Items it,
                                                         Entries pk, ChunkBufs cb,
                                                         unsigned long long* __restrict__ work,
                                                         const int* __restrict__ done) {
    __shared__ FwdLds s;
    __shared__ int s_slot[256];
    __shared__ int s_n;
    const int n = meta->n_items;
    for (int i0 = blockIdx.x; i0 < n; i0 += 256 * gridDim.x) {
        // items i0, i0 + gridDim.x, ...: neighbouring ones, which belong to
        // one tile, go to different workgroups
        const int64_t i = i0 + (int64_t)threadIdx.x * gridDim.x;
        bool mine = false;
        if (i < n) {
            const int y = it.rec[i].y;
            mine = (y & ITEM_LATE) && !done[y & ITEM_TILE];
        }
        __syncthreads();
        if (threadIdx.x == 0) s_n = 0;
        __syncthreads();
        if (mine) s_slot[atomicAdd(&s_n, 1)] = (int)i;
        __syncthreads();
        const int m = s_n;
        for (int j = 0; j < m; ++j)
            // chunked tiles only: no final pixels are written
            fwd_item<COUNT>(it.rec[s_slot[j]], W, H, tbx, 0.f, 0.f, 0.f, pk, nullptr, nullptr, nullptr, cb,
                            work, s);
    }
}

// Render-only forward, one workgroup per tile.  A tile rasterised in one
// piece is the forward above.  A chunked tile's chunks are rasterised in
// order, each from T = 1 as rasterize_forward_chunked_kernel does
// (.metal:2633-2741), and folded into the pixel's running state as the merge
// does (.metal:2746-2799): colour += chunk colour * T_running, T_running *=
// chunk T, final index = the chunk's last contributor, until T_running <=
// 1e-4.  A pixel past that cutoff takes no part in later chunks, and the
// workgroup stops once every pixel is past it: the chunks behind the cutoff,
// which only the backward's suffix sums read, are not rasterised.  The
// results are those of the chunk items plus the merge, bit for bit.
// At most 64 VGPRs (8 waves per SIMD; 71 unbounded, 7 waves): 1.5% more
// render FPS at config 3.
template <bool COUNT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_render_tiles(int W, int H, int tbx, float bg0,
                                                      float bg1, float bg2, Items it,
                                                      Entries pk, float* __restrict__ final_T,
                                                      int* __restrict__ final_idx,
                                                      float* __restrict__ out_img,
                                                      unsigned long long* __restrict__ work) {
    __shared__ FwdLds lds;
    const int4 rec = it.tile_rec[blockIdx.x];   // heaviest size class first
    const int t = rec.x, K = rec.y, s = rec.z, e = rec.w;
    const Px px = pixel_of(t, tbx, W, H);
    float fx = (float)px.j, fy = (float)px.i;
    asm volatile("" : "+v"(fx), "+v"(fy));
    const int tx0 = (t % tbx) * BLOCK, ty0 = (t / tbx) * BLOCK;
    unsigned ncl = 0, nwit = 0;
    float Tr = 1.f, R0 = 0.f, R1 = 0.f, R2 = 0.f;
    int li;
    if (K == 1) {
        li = s - 1;
        fwd_range<COUNT>(s, e, px.inside, fx, fy, tx0, ty0, pk, lds, Tr, R0, R1, R2, li, ncl, nwit);
    } else {
        li = -1;
        bool done = !px.inside;
        for (int k = 0; k < K; ++k) {
            if (__syncthreads_and(done)) break;
            const int cs = s + k * CHUNK, ce = min(cs + CHUNK, e);
            float T = 1.f, C0 = 0.f, C1 = 0.f, C2 = 0.f;
            int last = cs - 1;
            fwd_range<COUNT>(cs, ce, !done, fx, fy, tx0, ty0, pk, lds, T, C0, C1, C2, last, ncl, nwit);
            if (!done) {
                R0 = fmaf(C0, Tr, R0);
                R1 = fmaf(C1, Tr, R1);
                R2 = fmaf(C2, Tr, R2);
                Tr *= T;
                if (last >= 0) li = last;
                if (Tr <= 1e-4f) done = true;
            }
        }
    }
    add_work<COUNT>(work, ncl, nwit);
    if (!px.inside) return;
    const size_t pix = (size_t)px.i * W + px.j;
    final_T[pix] = Tr;
    final_idx[pix] = li;
    out_img[3 * pix + 0] = clamp01(fmaf(bg0, Tr, R0));
    out_img[3 * pix + 1] = clamp01(fmaf(bg1, Tr, R1));
    out_img[3 * pix + 2] = clamp01(fmaf(bg2, Tr, R2));
}

// Training forward of the chunked tiles in two launches: chunks k < P first;
// then, for a tile with more than P chunks, chunk k >= P only if some pixel
// of the tile still has a nonzero running transmittance after the first P
// (pT_P = T_0 T_1 ... T_{P-1}, multiplied in chunk order as the merge does).
// Where every pixel's pT_P is exactly 0, every later chunk j has pT_j = 0:
// its colour enters the suffix sums as pT_j * C_j = 0, it lies past every
// pixel's merge cutoff (T_running = pT <= 1e-4 before it), so the merge
// gives it index -1 and the backward skips it.  Its state would change no
// output bit, so it is not computed; the merge reads only the first P chunks
// of such a tile.  k_chunk_done marks those tiles.
__global__ __launch_bounds__(256) void k_chunk_done(int W, int H, int tbx,
                                                    const Meta* __restrict__ meta,
                                                    const int* __restrict__ chunked, Items it,
                                                    ChunkBufs cb, int* __restrict__ done) {
    constexpr int P = FWD_P;
    __shared__ int s_any;
    const int nch = meta->n_chunked_tiles;
    for (int b = blockIdx.x; b < nch; b += gridDim.x) {
        const int t = chunked[b];
        const int K = it.tile_K[t], i0 = it.tile_item0[t];
        if (K <= P) {
            if (threadIdx.x == 0) done[t] = 0;
            continue;
        }
        __syncthreads();     // the previous tile's s_any has been read
        if (threadIdx.x == 0) s_any = 0;
        __syncthreads();
        const int lp = threadIdx.x, lx = lp & 15, ly = lp >> 4;
        const int j = (t % tbx) * BLOCK + lx, i = (t / tbx) * BLOCK + ly;
        if (i < H && j < W) {
            // all P loads in flight, then the product in chunk order
            float c[P];
#pragma unroll
            for (int k = 0; k < P; ++k) c[k] = cb.cT[(size_t)(i0 + k) * TILE_PIX + lp];
            float pT = 1.f;
#pragma unroll
            for (int k = 0; k < P; ++k) pT *= c[k];
            if (pT != 0.f) s_any = 1;
        }
        __syncthreads();
        if (threadIdx.x == 0) done[t] = s_any ? 0 : 1;
    }
}

__global__ __launch_bounds__(256) void k_raster_merge(int W, int H, int tbx, float bg0,
                                                      float bg1, float bg2,
                                                      const Meta* __restrict__ meta,
                                                      const int* __restrict__ chunked, Items it,
                                                      float* __restrict__ final_T,
                                                      int* __restrict__ final_idx,
                                                      float* __restrict__ out_img, ChunkBufs cb,
                                                      int with_suffix, const int* __restrict__ done,
                                                      int P, int* __restrict__ live_end) {
    __shared__ int s_cut;
    if ((int)blockIdx.x >= meta->n_chunked_tiles) return;
    if (threadIdx.x == 0) s_cut = 0;
    __syncthreads();
    const int t = chunked[blockIdx.x];
    const int K = it.tile_K[t], i0 = it.tile_item0[t];
    // chunks with state: all K, or the first P of a tile whose later chunks
    // were not computed (they carry pT = 0 and change no output)
    const int Kc = (done && done[t]) ? min(K, P) : K;
    const int lp = threadIdx.x, lx = lp & 15, ly = lp >> 4;
    const int j = (t % tbx) * BLOCK + lx, i = (t / tbx) * BLOCK + ly;
    const bool inside = i < H && j < W;
    float Tr = 1.f, R0 = 0.f, R1 = 0.f, R2 = 0.f;
    int li = -1, cutoff = inside ? K : 0;
    // Chunks are folded front to back, stopping at an empty chunk or once
    // T <= 1e-4.  The state of MG chunks is loaded ahead of folding them
    // (every k < K is a valid chunk), so a tile with hundreds of chunks
    // costs one memory round trip per MG chunks instead of two per chunk.
    constexpr int MG = 8;
    bool stop = !inside;
    for (int k0 = 0; k0 < Kc && !stop; k0 += MG) {
        int cf[MG];
        float cT[MG], c0[MG], c1[MG], c2[MG];
#pragma unroll
        for (int u = 0; u < MG; ++u) {
            const int k = min(k0 + u, Kc - 1);
            const size_t o = (size_t)(i0 + k) * TILE_PIX + lp;
            cf[u] = cb.cidx[o];
            cT[u] = cb.cT[o];
            c0[u] = cb.cC[3 * o + 0];
            c1[u] = cb.cC[3 * o + 1];
            c2[u] = cb.cC[3 * o + 2];
        }
#pragma unroll
        for (int u = 0; u < MG; ++u) {
            const int k = k0 + u;
            if (k >= Kc || (cf[u] < 0 && k > 0)) {
                stop = true;
                break;
            }
            R0 = fmaf(c0[u], Tr, R0);
            R1 = fmaf(c1[u], Tr, R1);
            R2 = fmaf(c2[u], Tr, R2);
            Tr *= cT[u];
            if (cf[u] >= 0) li = cf[u];
            if (Tr <= 1e-4f) {
                cutoff = k + 1;
                stop = true;
                break;
            }
        }
    }
    // The chunks past a pixel's cutoff have no backward work there.  The items
    // from the largest cutoff of the tile's pixels on have none at all: the
    // backward stops at that item (live_end) and reads nothing of them, and
    // their indexes need no marking.
    const int wave_cut = wave_max_i(cutoff);
    if ((threadIdx.x & 63) == 0) atomicMax(&s_cut, wave_cut);
    __syncthreads();
    const int cut = s_cut;
    if (threadIdx.x == 0) live_end[t] = i0 + cut;
    if (!inside) return;
    for (int k = cutoff; k < cut; ++k) cb.cidx[(size_t)(i0 + k) * TILE_PIX + lp] = -1;
    const size_t pix = (size_t)i * W + j;
    final_T[pix] = Tr;
    final_idx[pix] = li;
    out_img[3 * pix + 0] = clamp01(fmaf(bg0, Tr, R0));
    out_img[3 * pix + 1] = clamp01(fmaf(bg1, Tr, R1));
    out_img[3 * pix + 2] = clamp01(fmaf(bg2, Tr, R2));
    if (!with_suffix) return;
    // prefix products of T and suffix sums of the chunk colours, each over
    // all chunks with state (the rest add pT * C = 0), with the loads of MG
    // chunks issued ahead of their stores
    float pT = 1.f;
    for (int k0 = 0; k0 < Kc; k0 += MG) {
        float t[MG];
#pragma unroll
        for (int u = 0; u < MG; ++u)
            t[u] = cb.cT[(size_t)(i0 + min(k0 + u, Kc - 1)) * TILE_PIX + lp];
#pragma unroll
        for (int u = 0; u < MG; ++u) {
            if (k0 + u >= Kc) break;
            cb.pT[(size_t)(i0 + k0 + u) * TILE_PIX + lp] = pT;
            pT *= t[u];
        }
    }
    float a0 = 0.f, a1 = 0.f, a2 = 0.f;
    for (int k1 = Kc - 1; k1 >= 0; k1 -= MG) {
        float pp[MG], q0[MG], q1[MG], q2[MG];
#pragma unroll
        for (int u = 0; u < MG; ++u) {
            const size_t o = (size_t)(i0 + max(k1 - u, 0)) * TILE_PIX + lp;
            pp[u] = cb.pT[o];
            q0[u] = cb.cC[3 * o + 0];
            q1[u] = cb.cC[3 * o + 1];
            q2[u] = cb.cC[3 * o + 2];
        }
#pragma unroll
        for (int u = 0; u < MG; ++u) {
            if (k1 - u < 0) break;
            const size_t o = (size_t)(i0 + k1 - u) * TILE_PIX + lp;
            cb.aC[3 * o + 0] = a0;
            cb.aC[3 * o + 1] = a1;
            cb.aC[3 * o + 2] = a2;
            a0 += pp[u] * q0[u];
            a1 += pp[u] * q1[u];
            a2 += pp[u] * q2[u];
        }
    }
}

// Inclusive product / sum scans over the 16 lanes of each row, of four values
// at once: the four chains fill the two wait states that a DPP read needs
// after the write of its source (the first pair of s_nop covers the caller's
// last write).  A lane without a source keeps its value.  All lanes must be
// active.
#define MSP_ROW_SCAN4(op, v)                                                              \
    asm volatile(                                                                        \
        "s_nop 1\n\t" MSP_ROW_SCAN4_STEP(op, "1") MSP_ROW_SCAN4_STEP(op, "2")            \
            MSP_ROW_SCAN4_STEP(op, "4") MSP_ROW_SCAN4_STEP(op, "8") "s_nop 1"            \
        : "+v"((v)[0]), "+v"((v)[1]), "+v"((v)[2]), "+v"((v)[3]))
#define MSP_ROW_SCAN4_STEP(op, n)                                              \
    op " %0, %0, %0 row_shr:" n " row_mask:0xf bank_mask:0xf\n\t"              \
    op " %1, %1, %1 row_shr:" n " row_mask:0xf bank_mask:0xf\n\t"              \
    op " %2, %2, %2 row_shr:" n " row_mask:0xf bank_mask:0xf\n\t"              \
    op " %3, %3, %3 row_shr:" n " row_mask:0xf bank_mask:0xf\n\t"

// The value of lane N of each row of 16, in all lanes of the row.
template <int N>
__device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(row_bcast<N>(__float_as_int(v)));
}
// The colour terms of a column's four pixels, lane X + 4 y of each row holding
// pixel y's (v0, v1, v2): rv[y] = v0 r + v1 g + v2 b, and (c0, c1, c2) = sum over
// y of (v0, v1, v2) fac[y], by multiply-adds in order.  The compiler does not
// fold a broadcast into a multiply-add by itself.  One block with the DPP wait
// states in front: the compiler's hazard logic does not look inside, and may
// place a copy of v0, v1 or v2 right before it.
#define MSP_COLOUR(op, d0, d1, d2, d3, v, s0, s1, s2, s3)                               \
    op " " d0 ", " v ", " s0 " row_newbcast:%[n0] row_mask:0xf bank_mask:0xf\n\t"       \
    op " " d1 ", " v ", " s1 " row_newbcast:%[n1] row_mask:0xf bank_mask:0xf\n\t"       \
    op " " d2 ", " v ", " s2 " row_newbcast:%[n2] row_mask:0xf bank_mask:0xf\n\t"       \
    op " " d3 ", " v ", " s3 " row_newbcast:%[n3] row_mask:0xf bank_mask:0xf\n\t"
#define MSP_COLOUR_RV(op, v, s) MSP_COLOUR(op, "%0", "%1", "%2", "%3", v, s, s, s, s)
#define MSP_COLOUR_SUM(op, d, v, f, n) op " " d ", " v ", " f " row_newbcast:%[" n "] row_mask:0xf bank_mask:0xf\n\t"
#define MSP_COLOUR_SUMS(op, f, n)                                                       \
    MSP_COLOUR_SUM(op, "%[c0]", "%[v0]", f, n) MSP_COLOUR_SUM(op, "%[c1]", "%[v1]", f, n) \
        MSP_COLOUR_SUM(op, "%[c2]", "%[v2]", f, n)
template <int X>
__device__ __forceinline__ void column_colours(float v0, float v1, float v2, float r, float g, float b,
                                               const float (&fac)[4], float (&rv)[4], float& c0, float& c1,
                                               float& c2) {
    asm("s_nop 1\n\t"
        MSP_COLOUR_RV("v_mul_f32_dpp", "%[v0]", "%[r]") MSP_COLOUR_RV("v_fmac_f32_dpp", "%[v1]", "%[g]")
        MSP_COLOUR_RV("v_fmac_f32_dpp", "%[v2]", "%[b]") MSP_COLOUR_SUMS("v_mul_f32_dpp", "%[f0]", "n0")
        MSP_COLOUR_SUMS("v_fmac_f32_dpp", "%[f1]", "n1") MSP_COLOUR_SUMS("v_fmac_f32_dpp", "%[f2]", "n2")
        MSP_COLOUR_SUMS("v_fmac_f32_dpp", "%[f3]", "n3")
        : "=&v"(rv[0]), "=&v"(rv[1]), "=&v"(rv[2]), "=&v"(rv[3]), [c0] "=&v"(c0), [c1] "=&v"(c1), [c2] "=&v"(c2)
        : [v0] "v"(v0), [v1] "v"(v1), [v2] "v"(v2), [r] "v"(r), [g] "v"(g), [b] "v"(b), [f0] "v"(fac[0]),
          [f1] "v"(fac[1]), [f2] "v"(fac[2]), [f3] "v"(fac[3]), [n0] "n"(X), [n1] "n"(X + 4), [n2] "n"(X + 8),
          [n3] "n"(X + 12));
}
// A point before which the compiler forms no broadcast of d (a loop's
// broadcasts are not hoisted into registers of their own).
__device__ __forceinline__ void keep_in_loop(int& d) { asm volatile("" : "+v"(d)); }
// The value of the lane before within the row; lane 0 gets first.
__device__ __forceinline__ float row_before(float v, float first) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(first), __float_as_int(v), 0x111,
                                                      0xF, 0xF, false));
}
__device__ __forceinline__ int row_max(int v) {
    v = max(v, __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
    v = max(v, __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true));    // quad_perm [2,3,0,1]
    v = max(v, __builtin_amdgcn_mov_dpp(v, 0x124, 0xF, 0xF, true));   // row_ror:4
    return max(v, __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true));  // row_ror:8
}

// f(0), f(1), ... f(N - 1) with the index as a compile-time constant.
template <typename F, int... P>
__device__ __forceinline__ void for_each_of(F& f, std::integer_sequence<int, P...>) {
    (f(std::integral_constant<int, P>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void for_each_to(F f) {
    for_each_of(f, std::make_integer_sequence<int, N>{});
}

// Window of a backward wave: up to WIN entries that reach its quadrant, and
// the dummy behind them; their gradient sums; the rows' lists of window slots.
// 8.2 KB; the 119 vector registers allow four waves a SIMD (five, at 96
// registers with spills, measured 2% slower; windows of 128 entries the same).
constexpr int WIN = 96;
struct BwdLds {
    float4 geo[WIN + 1];      // x, y, conic a, b
    float4 col[WIN + 1];      // conic c, opacity, clamped r, g
    float2 aux[WIN + 1];      // clamped b, -entry index (bits)
    int gid[WIN];             // gaussian
    float4 sa[WIN], sb[WIN];  // the sums 0..3 and 4..7 of gacc's nine
    float sc[WIN];            // and the last
    uint8_t rows[WIN];        // rows an entry is wanted by
    uint8_t list[4][WIN];
};

// The state of a row's 16 pixels, pixel p of the row's block in register p
// (the same in all lanes of the row): transmittance behind and E (below).
struct RowState {
    float T[16], E[16];
};

// This lane's entry and its sums over the pixels of the row's block.
struct EntrySums {
    float s0, s1, s2, s11, s12, s22;   // v_sigma, v_sigma (dx, dy, dx^2, dx dy, dy^2)
    float c0, c1, c2;                  // fac v_out
};

// Column X of the row's block (pixels X, X + 4, X + 8, X + 12; column 3 comes
// first), all 16 entries of the group at once: lane l of a row holds the row's
// l-th entry, deepest first.  vo0..2 and bf are per pixel, in the pixel's lane: the pixel takes the
// entries up to index bf (tested as the sign of bf - index, formed by an add:
// a subtraction that takes its subtrahend through DPP, v_subrev, was measured
// to broadcast the other operand).
template <bool COUNT, int X>
__device__ __forceinline__ void bwd_column(float4 g, float4 c, float blue, int nidx, float fx0,
                                           const float* dy, const float* cy2, float vo0, float vo1,
                                           float vo2, int bf, RowState& st, EntrySums& es,
                                           unsigned& ngrad) {
    const float dx = g.x - (fx0 + (float)X);
    const float dx2 = dx * dx, bx = g.w * dx;
    float ag[4], ra[4], P[4], Tn[4], fac[4], RV[4], S[4];
    auto pixel = [&](auto yc) {
        constexpr int y = decltype(yc)::value, p = 4 * y + X;
        const float sigma = fmaf(0.5f, fmaf(g.z, dx2, cy2[y]), bx * dy[y]);
        const float alpha = c.y * exp_neg_raster(sigma_clamp(sigma));
        // a gradient flows where the entry is not behind the pixel's last
        // contributor and 1/255 <= alpha < 0.999 (one unsigned compare of the
        // bits; NaN is above); elsewhere alpha = 0 leaves the state as it is
        // (1 / (1 - 0) = 1) and makes every term zero
        const unsigned behind = (unsigned)(row_bcast<p>(bf) + nidx) & 0x80000000u;
        const bool ok = ((__float_as_uint(alpha) - 0x3B808081u) | behind) < 0x3F7FBE77u - 0x3B808081u;
        ag[y] = ok ? alpha : 0.f;
        if (COUNT) ngrad += (unsigned)__popcll(wave_ballot(ok));
        // hardware reciprocal (1 ulp, exact at 1): the backward is compared
        // with a tolerance
        P[y] = ra[y] = __builtin_amdgcn_rcpf(1.f - ag[y]);
    };
    for_each_to<4>(pixel);
    MSP_ROW_SCAN4("v_mul_f32_dpp", P);
    auto terms = [&](auto yc) {
        constexpr int y = decltype(yc)::value, p = 4 * y + X;
        Tn[y] = st.T[p] * P[y];
        fac[y] = ag[y] * Tn[y];
        st.T[p] = row_bcast<15>(Tn[y]);
    };
    for_each_to<4>(terms);
    float c0, c1, c2;
    column_colours<X>(vo0, vo1, vo2, c.z, c.w, blue, fac, RV, c0, c1, c2);
#pragma unroll
    for (int y = 0; y < 4; ++y) S[y] = fac[y] * RV[y];
    MSP_ROW_SCAN4("v_add_f32_dpp", S);
    float s = 0.f, t = 0.f, u = 0.f;     // the column's sums of v, v dy and v dy^2
    auto sums = [&](auto yc) {
        constexpr int y = decltype(yc)::value, p = 4 * y + X;
        const float Ei = st.E[p] + S[y];
        const float E = row_before(Ei, st.E[p]);    // behind this entry
        st.E[p] = row_bcast<15>(Ei);
        // v_alpha = sum_k (r_k Tn - (B_k + T_final bg_k) ra) v_out_k
        const float v_alpha = fmaf(Tn[y], RV[y], -ra[y] * E);
        const float v = -ag[y] * v_alpha;
        const float vy = v * dy[y];
        s = y == 0 ? v : s + v;
        t = y == 0 ? vy : t + vy;
        u = y == 0 ? vy * dy[y] : fmaf(vy, dy[y], u);
    };
    for_each_to<4>(sums);
    // sums of four pixels, then of four columns (and then of four rows, in the
    // window's sums): a term passes nine additions.  In one chain over the 16
    // pixels it passed 18, and 64 equal terms came out up to 4.1 units of 2^-24 off
    // (now 1.4; the same time: 1225.6 and 1226.7 us a step of 1.5M gaussians).
    constexpr bool first = X == 3;
    es.s0 = first ? s : es.s0 + s;
    es.s1 = first ? s * dx : fmaf(s, dx, es.s1);
    es.s11 = first ? s * dx2 : fmaf(s, dx2, es.s11);
    es.s12 = first ? t * dx : fmaf(t, dx, es.s12);
    es.s2 = first ? t : es.s2 + t;
    es.s22 = first ? u : es.s22 + u;
    es.c0 = first ? c0 : es.c0 + c0;
    es.c1 = first ? c1 : es.c1 + c1;
    es.c2 = first ? c2 : es.c2 + c2;
    // one column at a time: interleaved columns would need more registers
    // than the four pixels of one, which already fill the DPP wait states,
    // and so would sums put off until they are used
    asm volatile("" : "+v"(es.s0), "+v"(es.s1), "+v"(es.s2), "+v"(es.s11), "+v"(es.s12), "+v"(es.s22),
                 "+v"(es.c0), "+v"(es.c1), "+v"(es.c2));
    __builtin_amdgcn_sched_barrier(0);
}

// The backward turns the forward's roles round: a row of 16 lanes takes 16
// entries of its block's list at once, one per lane and deepest first, and
// goes through the block's 16 pixels one after the other.  What a pixel
// carries from entry to entry (the transmittance behind the entry and the
// colour accumulated behind it) becomes a product and a sum scan over the
// row's lanes (four DPP steps each), and an entry's gradient sums over the
// pixels stay in its lane's registers: no reduction over lanes.
// One wave is a workgroup of its own, for one quadrant of a record: no
// barriers, and a heavy quadrant holds up nothing but itself.  It puts together
// a window of up to WIN entries that reach its quadrant, gathers them and lists
// them by row, walks them, and adds the window's sums to gacc with consecutive
// lanes on consecutive floats.  (Gathered and listed 64 entries of the tile at a
// time, most of them unwanted, 100k needles of sd 110 pixels at 1297x840, whose
// rectangles cover tiles that they miss, took 734 us, now 584, where lane =
// pixel took 519; the whole step 1941, 1796 and 1797.)
// The window's sums are kept in LDS; an LDS float atomic takes 193 cycles of
// the CU for a wave whatever its addresses (a plain store 7.5), so each row
// adds its sums in turn with ordinary loads and stores (entries of one row are
// distinct, those of different rows are not).
// Bound: the vector units (294M instructions in a step of 1.5M trained gaussians
// at 1297x840: four cycles each are 0.48 of its 0.53 ms).  Per (entry, pixel)
// pair of lanes: about 57 vector instructions, no scalar ones and no LDS access
// (75, 6 and 3 with the windows, lists and sums around them), where lane = pixel
// took 65, 11 and 11; a block of 4 x 4 pixels leaves fewer pairs
// without a gradient than an 8 x 8 quadrant (2.10M wave steps against 2.75M).
// Measured against lane = pixel with 8 x 8 quadrants: 10k gaussians at 256x256
// 32 -> 16 us, 120k at 324x210 60 -> 37 us, 1M in a blob at 2594x1680 592 ->
// 558 us, 1.5M at 1297x840 281 -> 284 us.  The colour terms on the matrix cores
// (v_mfma_f32_4x4x1) instead of by DPP: the same time, from register spills.
// COUNT: count the wave's evaluated entries and gradient pairs into work
// (a launch without counters runs the variant that does not count).
template <bool COUNT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void k_raster_bwd(
    int W, int H, int tbx, float bg0, float bg1, float bg2, const Meta* __restrict__ meta, Items it,
    Entries pk, const float* __restrict__ final_T, const int* __restrict__ final_idx, ChunkBufs cb,
    const int* __restrict__ live_end, const float* __restrict__ v_out,
    float* __restrict__ gacc, unsigned long long* __restrict__ work, LossFold lf) {
    __shared__ BwdLds s;
    // Workgroup 0 folds the loss partials of the SSIM tiles and takes no
    // item: dispatched first, it runs beside the heaviest items instead of
    // at the end of the launch.
    static_assert(sizeof(s.sa) >= 3 * 64 * sizeof(double), "loss fold area");
    if (blockIdx.x == 0) {
        if (lf.part) loss_fold(lf, reinterpret_cast<double*>(s.sa));
        return;
    }
    // items in launch order (heaviest size class first); the four quadrants of
    // an item are eight workgroups apart, so they run on one XCD at about the
    // same time and gather the entries' records through one L2
    const int wg = (int)blockIdx.x - 1;
    const int bi = (wg >> 5) * 8 + (wg & 7), w = (wg >> 3) & 3;
    if (bi >= meta->n_groups) return;
    const int4 rec = it.bwd_rec[bi];
    const bool multi = (rec.y & ITEM_MULTI) != 0;
    const int t = rec.y & ITEM_TILE;
    const int item_end = multi ? live_end[t] : rec.x + 1;   // (of a chunked tile) items with work
    if (rec.x >= item_end) return;
    const int lane = threadIdx.x, i = lane & 15, row = lane >> 4;
    const Px px = pixel_at(t, tbx, W, H, 64 * w + lane);

    const size_t pix = (size_t)px.i * W + px.j;
    if (lane == 0) {
        s.geo[WIN] = s.col[WIN] = make_float4(0.f, 0.f, 0.f, 0.f);
        s.aux[WIN] = make_float2(0.f, 0.f);
    }
    for (int k = lane; k < WIN; k += 64) {
        s.sa[k] = s.sb[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        s.sc[k] = 0.f;
    }
    // the pixel whose lane this is lies in column i & 3, row i >> 2 of its
    // block, whose first pixel is (fx0, fy0)
    const float fx0 = (float)(px.j - (i & 3)), fy0 = (float)(px.i - (i >> 2));
    unsigned ngrad = 0;     // pairs of this wave that carry a gradient (wave-uniform)
    unsigned nwit = 0;      // entries this wave evaluated (wave-uniform)
    float Tfin = 1.f, vo0 = 0.f, vo1 = 0.f, vo2 = 0.f;
    if (px.inside) {
        Tfin = final_T[pix];
        vo0 = v_out[3 * pix + 0];
        vo1 = v_out[3 * pix + 1];
        vo2 = v_out[3 * pix + 2];
    }

    // the record's chunks one after the other (a tile in one piece is one);
    // each starts from its own state
    int item = rec.x;
    for (int cs = rec.z, ce; cs < rec.w && item < item_end; cs = ce, ++item) {
    ce = multi ? min(cs + CHUNK, rec.w) : rec.w;
    float T = Tfin, B0 = 0.f, B1 = 0.f, B2 = 0.f;
    // bf = cs - 1 for pixels outside the image: no entry passes e_idx <= bf
    int bf = cs - 1;
    const size_t chunk_pix = (size_t)item * TILE_PIX + px.lp;
    if (px.inside) bf = multi ? cb.cidx[chunk_pix] : final_idx[pix];
    // the last contributor of each row's pixels (wave-uniform)
    const int rbf = row_max(bf);
    const int row_bf[4] = {__builtin_amdgcn_readlane(rbf, 0), __builtin_amdgcn_readlane(rbf, 16),
                           __builtin_amdgcn_readlane(rbf, 32), __builtin_amdgcn_readlane(rbf, 48)};
    int top = min(ce - 1, max(max(row_bf[0], row_bf[1]), max(row_bf[2], row_bf[3])));
    if (top < cs) continue;
    // the next 64 entries' block masks and ids, loaded ahead of their use
    int idx = top - lane;
    unsigned mask = idx >= cs ? pk.bmask[idx] : 0u;
    int gid = idx >= cs ? (int)pk.ids[idx] : 0;
    if (px.inside && multi) {
        T = cb.pT[chunk_pix] * cb.cT[chunk_pix];
        B0 = cb.aC[3 * chunk_pix + 0];
        B1 = cb.aC[3 * chunk_pix + 1];
        B2 = cb.aC[3 * chunk_pix + 2];
    }
    // The colour terms of v_alpha enter only as sum_k v_out_k (...)_k:
    // D = sum_k v_out_k B_k (accumulated colour behind) and TB = sum_k
    // v_out_k T_final bg_k are carried instead of the three channels.
    // E = D + TB, the two carried together: D changes, TB does not
    const float TB = fmaf(Tfin * bg2, vo2, fmaf(Tfin * bg1, vo1, (Tfin * bg0) * vo0));
    const float E = fmaf(B2, vo2, fmaf(B1, vo1, B0 * vo0)) + TB;
    RowState st;
    auto spread = [&](auto pc) {
        constexpr int p = decltype(pc)::value;
        st.T[p] = row_bcast<p>(T);
        st.E[p] = row_bcast<p>(E);
    };
    for_each_to<16>(spread);
    const int bf_low = min(min(row_bf[0], row_bf[1]), min(row_bf[2], row_bf[3]));
    while (top >= cs) {
        // the window's entries, from 64 of the list at a time while they fit
        int nw = 0;
        while (top >= cs) {
            // rows this entry is wanted by: its block is reached, and it is
            // not behind the last contributor of the row's pixels
            unsigned m = (mask >> (4 * w)) & 15u;
            if (top > bf_low) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (idx > row_bf[r]) m &= ~(1u << r);
            }
            const uint64_t in = wave_ballot(m != 0u);
            const int cnt = __popcll(in);
            if (nw + cnt > WIN) break;
            if (m) {
                const int slot = nw + lanes_below(in);
                s.rows[slot] = (uint8_t)m;
                s.gid[slot] = gid;
                s.aux[slot].y = __int_as_float(-idx);
            }
            nw += cnt;
            top -= 64;
            idx = top - lane;
            mask = idx >= cs ? pk.bmask[idx] : 0u;
            gid = idx >= cs ? (int)pk.ids[idx] : 0;
        }
        __builtin_amdgcn_wave_barrier();
        // their records and the rows' lists, 64 of the window at a time
        int n[4] = {0, 0, 0, 0};
        for (int k0 = 0; k0 < nw; k0 += 64) {
            const int slot = k0 + lane;
            unsigned m = 0;
            if (slot < nw) {
                m = s.rows[slot];
                const float4* r = pk.rec + 4 * (size_t)s.gid[slot];
                const float4 g = r[0];
                const float4 c = r[1];
                const float braw = r[2].x;
                s.geo[slot] = g;
                s.col[slot] = make_float4(c.x, c.y, fmaxf(c.z + 0.5f, 0.f), fmaxf(c.w + 0.5f, 0.f));
                s.aux[slot].x = fmaxf(braw + 0.5f, 0.f);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint64_t b = wave_ballot((m >> r) & 1u);
                const int at = n[r] + lanes_below(b);
                if (lane_of(b)) s.list[r][at] = (uint8_t)slot;
                n[r] += __popcll(b);
            }
        }
        __builtin_amdgcn_wave_barrier();
        const int longest = max(max(n[0], n[1]), max(n[2], n[3]));
        const int mine = row == 0 ? n[0] : row == 1 ? n[1] : row == 2 ? n[2] : n[3];
        for (int p0 = 0; p0 < longest; p0 += 16) {
            const int slot = p0 + i < mine ? (int)s.list[row][p0 + i] : WIN;
            const float4 g = s.geo[slot];
            const float4 c = s.col[slot];
            const float blue = s.aux[slot].x;
            const int nidx = __float_as_int(s.aux[slot].y);
            if (COUNT) nwit += min(longest - p0, 16);
            float dy[4], cy2[4];
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                dy[y] = g.y - (fy0 + (float)y);
                cy2[y] = c.x * dy[y] * dy[y];
            }
            EntrySums es;
            keep_in_loop(bf);
            bwd_column<COUNT, 3>(g, c, blue, nidx, fx0, dy, cy2, vo0, vo1, vo2, bf, st, es, ngrad);
            bwd_column<COUNT, 2>(g, c, blue, nidx, fx0, dy, cy2, vo0, vo1, vo2, bf, st, es, ngrad);
            bwd_column<COUNT, 1>(g, c, blue, nidx, fx0, dy, cy2, vo0, vo1, vo2, bf, st, es, ngrad);
            bwd_column<COUNT, 0>(g, c, blue, nidx, fx0, dy, cy2, vo0, vo1, vo2, bf, st, es, ngrad);
            // v_xy = v_sigma (a dx + b dy, b dx + c dy) and v_conic = v_sigma
            // / 2 (dx^2, dx dy, dy^2) are linear in these moments with the
            // gaussian's own conic, the same in every tile: the projection
            // backward applies the conic once per gaussian.  The opacity
            // (logit) term is -v_sigma (1 - o).  v_rgb of a channel whose raw
            // colour + 0.5 < 0 is dropped by its consumers.
            const float so = es.s0 * (c.y - 1.f);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (row == r && slot < WIN) {
                    float4 a = s.sa[slot], b = s.sb[slot];
                    a.x += es.s1;
                    a.y += es.s2;
                    a.z += es.s11;
                    a.w += es.s12;
                    b.x += es.s22;
                    b.y += es.c0;
                    b.z += es.c1;
                    b.w += es.c2;
                    s.sa[slot] = a;
                    s.sb[slot] = b;
                    s.sc[slot] += so;
                }
                __builtin_amdgcn_wave_barrier();
            }
        }
        // the window's sums, consecutive lanes taking consecutive floats of a
        // gaussian's nine; entries without a gradient add nothing
        for (int k = lane; k < 9 * nw; k += 64) {
            const int e = (int)((unsigned)k / 9u), q = k - 9 * e;
            float* a = q < 8 ? reinterpret_cast<float*>(q < 4 ? s.sa : s.sb) + 4 * e + (q & 3) : s.sc + e;
            const float v = *a;
            *a = 0.f;
            if (v != 0.f) atomicAdd(gacc + 9 * (size_t)s.gid[e] + q, v);
        }
        __builtin_amdgcn_wave_barrier();
    }
    }
    if (COUNT && work) {
        unsigned long long* ws = work_slot(work);
        if (lane == 0 && ngrad) atomicAdd(ws + 1, (unsigned long long)ngrad);
        if (lane == 0 && nwit) atomicAdd(ws + 3, (unsigned long long)nwit);
    }
}

// Algorithmic work of the most recent forward (+ backward): one thread per
// pixel walks its item's entries in the order of the per-pixel loops of the
// reference kernels, without block culling or lockstep, and counts
// (pixel, entry) pairs: forward tested / sigma in range / composited,
// backward tested / sigma in range / carrying a gradient.  The counts
// define the algorithmic flops of the roofline; they change no state.
__global__ __launch_bounds__(256) void k_raster_work(int W, int H, int tbx,
                                                     const Meta* __restrict__ meta, Items it,
                                                     Entries pk,
                                                     const int* __restrict__ final_idx,
                                                     ChunkBufs cb,
                                                     const int* __restrict__ live_end,
                                                     unsigned long long* __restrict__ out) {
    if ((int)blockIdx.x >= meta->n_items) return;
    const int4 rec = it.rec[blockIdx.x];
    const int item = rec.x, t = rec.y & ITEM_TILE, cs = rec.z, ce = rec.w;
    const Px px = pixel_of(t, tbx, W, H);
    unsigned n[6] = {0u, 0u, 0u, 0u, 0u, 0u};
    if (px.inside) {
        const float fx = (float)px.j, fy = (float)px.i;
        float T = 1.f;
        for (int i = cs; i < ce; ++i) {
            ++n[0];
            const float4* r = pk.rec + 4 * (size_t)pk.ids[i];
            const float4 g = r[0];
            const float4 c = r[1];
            const float dx = g.x - fx, dy = g.y - fy;
            const float sigma = fmaf(0.5f, fmaf(g.z, dx * dx, c.x * dy * dy), g.w * dx * dy);
            if (!(sigma < 0.f || sigma >= 5.55f)) ++n[1];
            const float alpha = fminf(0.999f, c.y * exp_neg_raster(sigma_clamp(sigma)));
            if (alpha < 1.f / 255.f) continue;
            const float nT = T * (1.f - alpha);
            if (nT <= 1e-4f) break;
            ++n[2];
            T = nT;
        }
        const int bf = !(rec.y & ITEM_MULTI) ? final_idx[(size_t)px.i * W + px.j]
                       : item < live_end[t]  ? cb.cidx[(size_t)item * TILE_PIX + px.lp]
                                             : -1;
        for (int i = min(bf, ce - 1); i >= cs; --i) {
            ++n[3];
            const float4* r = pk.rec + 4 * (size_t)pk.ids[i];
            const float4 g = r[0];
            const float4 c = r[1];
            const float dx = g.x - fx, dy = g.y - fy;
            const float sigma = fmaf(0.5f, fmaf(g.z, dx * dx, c.x * dy * dy), g.w * dx * dy);
            if (!(sigma < 0.f || sigma >= 5.55f)) ++n[4];
            const float alpha = fminf(0.999f, c.y * exp_neg_raster(sigma_clamp(sigma)));
            if (alpha < 1.f / 255.f || !(alpha < 0.999f)) continue;
            ++n[5];
        }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        unsigned long long v = n[k];
        for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
        if ((threadIdx.x & 63) == 0) atomicAdd(&out[k], v);
    }
}

}  // namespace

void launch_raster_work(hipStream_t s, const CamParams& p, int64_t max_items, const Meta* meta,
                        Items it, Entries pk, const int* final_idx,
                        ChunkBufs cb, const int* live_end, unsigned long long* out) {
    if (max_items <= 0) return;
    hipLaunchKernelGGL(k_raster_work, dim3((unsigned)max_items), dim3(256), 0, s, p.W, p.H, p.tbx,
                       meta, it, pk, final_idx, cb, live_end, out);
}

void launch_raster_fwd(hipStream_t s, const CamParams& p, int64_t max_items, const Meta* meta,
                       Items it, Entries pk, float* final_T, int* final_idx,
                       float* out_img, ChunkBufs cb, unsigned long long* work, const int* chunked,
                       int* done) {
    if (max_items <= 0) return;
    // chunks 0 .. FWD_P - 1 of every tile, then the tiles' later chunks that
    // k_chunk_done does not mark as past an all-zero running transmittance
    // the counting variants only when pair counters are asked for
    if (work)
        hipLaunchKernelGGL(k_raster_fwd<true>, dim3((unsigned)max_items), dim3(256), 0, s, p.W, p.H,
                           p.tbx, p.bg[0], p.bg[1], p.bg[2], meta, it, pk, final_T,
                           final_idx, out_img, cb, work);
    else
        hipLaunchKernelGGL(k_raster_fwd<false>, dim3((unsigned)max_items), dim3(256), 0, s, p.W, p.H,
                           p.tbx, p.bg[0], p.bg[1], p.bg[2], meta, it, pk, final_T,
                           final_idx, out_img, cb, work);
    const int T = p.tbx * p.tby;
    hipLaunchKernelGGL(k_chunk_done, dim3((unsigned)std::min(T, 256)), dim3(256), 0, s, p.W, p.H,
                       p.tbx, meta, chunked, it, cb, done);
    const dim3 tg((unsigned)std::min<int64_t>(max_items, 1024));
    if (work)
        hipLaunchKernelGGL(k_raster_fwd_tail<true>, tg, dim3(256), 0, s, p.W, p.H, p.tbx, meta, it,
                           pk, cb, work, (const int*)done);
    else
        hipLaunchKernelGGL(k_raster_fwd_tail<false>, tg, dim3(256), 0, s, p.W, p.H, p.tbx, meta, it,
                           pk, cb, work, (const int*)done);
}

void launch_render_tiles(hipStream_t s, const CamParams& p, Items it, Entries pk, float* final_T, int* final_idx, float* out_img,
                         unsigned long long* work) {
    const int T = p.tbx * p.tby;
    if (T <= 0) return;
    if (work)
        hipLaunchKernelGGL(k_render_tiles<true>, dim3((unsigned)T), dim3(256), 0, s, p.W, p.H, p.tbx,
                           p.bg[0], p.bg[1], p.bg[2], it, pk, final_T, final_idx, out_img,
                           work);
    else
        hipLaunchKernelGGL(k_render_tiles<false>, dim3((unsigned)T), dim3(256), 0, s, p.W, p.H, p.tbx,
                           p.bg[0], p.bg[1], p.bg[2], it, pk, final_T, final_idx, out_img,
                           work);
}

void launch_raster_merge(hipStream_t s, const CamParams& p, const Meta* meta, const int* chunked,
                         Items it, float* final_T, int* final_idx, float* out_img, ChunkBufs cb,
                         bool with_suffix, const int* done, int* live_end) {
    const int T = p.tbx * p.tby;
    hipLaunchKernelGGL(k_raster_merge, dim3(T), dim3(256), 0, s, p.W, p.H, p.tbx, p.bg[0], p.bg[1],
                       p.bg[2], meta, chunked, it, final_T, final_idx, out_img, cb,
                       with_suffix ? 1 : 0, done, FWD_P, live_end);
}

void launch_raster_bwd(hipStream_t s, const CamParams& p, int64_t max_groups, const Meta* meta,
                       Items it, Entries pk, const float* final_T,
                       const int* final_idx, ChunkBufs cb, const int* live_end, const float* v_out,
                       float* gacc, unsigned long long* work, const LossFold& lf) {
    // workgroup 0 folds the loss, the others take the records' quadrants (eight
    // records at a time)
    const int64_t g = (std::max<int64_t>(max_groups, 0) + 7) / 8 * 32 + 1;
    if (work)
        hipLaunchKernelGGL(k_raster_bwd<true>, dim3((unsigned)g), dim3(64), 0, s, p.W, p.H,
                           p.tbx, p.bg[0], p.bg[1], p.bg[2], meta, it, pk, final_T,
                           final_idx, cb, live_end, v_out, gacc, work, lf);
    else
        hipLaunchKernelGGL(k_raster_bwd<false>, dim3((unsigned)g), dim3(64), 0, s, p.W, p.H,
                           p.tbx, p.bg[0], p.bg[1], p.bg[2], meta, it, pk, final_T,
                           final_idx, cb, live_end, v_out, gacc, work, lf);
}

}  // namespace msp
