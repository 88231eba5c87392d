// kernels.hpp — launch interface between the C-ABI orchestration (context.hip)
// and the kernel translation units.  Host-callable launchers only.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace msp {

// Camera / render constants shared by projection, binning and raster.
struct CamParams {
    int N;
    float glob_scale;
    float vm[16];
    float pm[16];
    float fx, fy, cx, cy;
    int W, H;
    int tbx, tby;
    float clip;
    uint32_t key0;   // depth keys: the depth's bits less these (the near plane's, if it is positive)
    int degree;          // SH degree of the stored coefficients
    int dtu;             // degrees_to_use (clamped to degree)
    int rest_per;        // floats per gaussian in features_rest
    float cam[3];
    float bg[3];
};

// Per-gaussian outputs of the projection (internal layout).  One 64-byte
// record per gaussian so that the per-intersection gathers touch one cache
// line:  rec[4g+0] = (x, y, conic_a, conic_b)
//        rec[4g+1] = (conic_c, sigmoid(opacity), r, g)   raw SH colour
//        rec[4g+2] = (b, extent_x, extent_y, depth)
//        rec[4g+3] = (view direction normalize(p - cam), 0)
struct GaussOut {
    float4* rec;
    int* radii;
    int* radii_out;      // optional second copy of the radii (the caller's), or null
    int* tiles_hit;
    uint2* rect;         // tile rectangle: (x0 | y0 << 16, x1 | y1 << 16), 0 when culled
};

// Tile-sorted entries: ids[i] is the gaussian of entry i; the rasteriser
// gathers its projection record rec[4 id .. 4 id + 2] (one 64-byte line).
struct Entries {
    const uint32_t* ids;
    const float4* rec;
    // The 16-bit block mask of each entry, which the training forward computes
    // for every entry it stages, read back by the backward (which walks only
    // entries up to the last contributor, all of them staged by the forward)
    // instead of computing it again.
    uint16_t* bmask;
};

// Work items of the rasteriser, one per (tile, chunk).  The kernels take one
// record each, in launch order (heaviest size class first), so that a
// workgroup knows its range after a single load:
//   rec[slot]      = (item, tile | flags, first entry, end entry)
//   tile_rec[slot] = (tile, chunks, first entry, end entry)
//   bwd_rec[slot] = (first item, tile | flags, first entry, end entry) of the
//     backward: a whole tile, or up to BWD_GROUP consecutive chunks of one
// item numbers count the chunks tile by tile (tile_item0).
constexpr int ITEM_MULTI = 1 << 30;              // the tile has more than one chunk
constexpr int ITEM_LATE = (int)0x80000000u;      // chunk FWD_P or later of its tile
constexpr int ITEM_TILE = ITEM_MULTI - 1;
struct Items {
    int4* rec;
    int4* tile_rec;
    int4* bwd_rec;
    int* tile_K;         // chunks per tile
    int* tile_item0;     // first item of each tile
    int* cls;            // 6 x 32 counters of the size classes (items, tiles, groups; counts, fills)
};

// Host-visible summary written by the tile scan.
struct Meta {
    int64_t total_isect;
    int32_t max_count;
    int32_t n_items;
    int32_t n_chunked_tiles;   // tiles with more than one chunk
    int32_t n_large;           // unused (0)
    int32_t n_huge;            // unused (0)
    int32_t n_groups;          // records of the backward
};

// Tile lists written by the tile scan (order within a list is arbitrary).
struct TileLists {
    int* chunked;
    int* large;
    int* huge;
};


// Per-pixel chunk state, indexed by item * 256 + local pixel.
struct ChunkBufs {
    float* cT;
    float* cC;           // x3
    int* cidx;
    float* pT;
    float* aC;           // x3
};

// Counters of the projection: ISECT_SLOTS slots of u64 counters ISECT_STRIDE
// u64 apart (one 128-byte line each); a slot's first counts (gaussian, tile)
// pairs, the second (gaussian, super-tile) references, the third is set where
// a depth key takes more than FAR_BITS bits; the totals over the slots are
// formed by the first kernel of the depth sort (SlotSum) for the host.
constexpr int FAR_BITS = 27;
constexpr int ISECT_SLOTS = 64;
constexpr int ISECT_STRIDE = 16;
constexpr size_t ISECT_BYTES = (size_t)ISECT_SLOTS * ISECT_STRIDE * 8;
void launch_project_fwd(hipStream_t s, const CamParams& p, const float* means,
                        const float* scales, const float* quats, const float* f_dc,
                        const float* f_rest, const float* opac_logits, GaussOut go,
                        uint32_t* dkey, uint32_t* dval, float* gacc,
                        unsigned long long* total_isect);

// Block totals and radix sort (radix.hip).
constexpr int SCAN_BLOCK = 1024;   // elements per scan block
int64_t scan_block_count(int64_t n);
// Above this many 1024-element blocks a scan runs its block totals through a
// one-workgroup scan; up to it, each block adds up the totals before it.
constexpr int SCAN_DIRECT_BLOCKS = 2048;
// The first half of a scan: the totals of the 1024-element blocks of in,
// turned into exclusive block offsets when there are more than
// SCAN_DIRECT_BLOCKS blocks (the consumer then reads tot[b] directly).
void launch_block_totals(hipStream_t s, const int* in, int64_t n, int* tot);
int64_t radix_temp_ints(int64_t n);
// Optional side job of a sort's first kernel, for the depth order: its
// workgroup 0 sums the projection's ISECT_SLOTS counter pairs and writes the
// two totals to *out (coherent host memory) as one 64-bit word,
// totals_word(I, R), which the host polls.
struct SlotSum {
    const unsigned long long* slots = nullptr;
    unsigned long long* out = nullptr;
    int* far = nullptr;   // gets 1 if a depth key takes more than FAR_BITS bits, else 0
};
// Bit 63 set (so that a zeroed word means "not yet"), bit 62 if a depth key
// takes more than FAR_BITS bits, the intersection total in bits 31..61 and the
// reference total in bits 0..30, each saturated at 2^31 - 1.
__host__ __device__ inline unsigned long long totals_word(unsigned long long i, unsigned long long r, bool far) {
    const unsigned long long cap = 0x7FFFFFFFull;
    return (1ull << 63) | ((far ? 1ull : 0ull) << 62) | ((i < cap ? i : cap) << 31) | (r < cap ? r : cap);
}
// Optional epilogue of a sort's last pass, for the depth order: output
// position i also gets rs[i] = rect[value] and cnt[i] = the super-tile count
// of that rectangle (both zero at the positions of a culling sort's culled
// tail).
struct RectGather {
    const uint2* rect = nullptr;
    uint2* rs = nullptr;
    int* cnt = nullptr;
    const int* skip = nullptr;   // nothing is written where this holds nonzero
};
// Up to RANK_MAX keys are ordered by ranking (all pairs compared) instead.  A
// 256x256 render took, sorted / ranked: 98 / 44 us for 2k gaussians, 115 / 63
// for 10k, 133 / 93 for 20k, 149 / 129 for 28k, 155 / 156 for 32k; the line
// lies below the crossing.
// vout, rg: the values, rectangles and counts in order; tot: the counts' block
// totals, as launch_block_totals leaves them; rank: n ints, zero between calls.
constexpr int RANK_MAX = 24 * SCAN_BLOCK;
void launch_rank_order(hipStream_t s, const uint32_t* key, const uint32_t* val, int n, int* rank,
                       uint32_t* vout, int* tot, const RectGather& rg, const SlotSum& ss);
bool launch_radix_sort(hipStream_t s, uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1,
                       int64_t n, int bits, int* temp, const RectGather* rg = nullptr,
                       const SlotSum* ss = nullptr, int* edge0 = nullptr, int* edge1 = nullptr,
                       bool cull = false);
void launch_radix_far(hipStream_t s, const uint32_t* ki, const uint32_t* vi, uint32_t* ko, uint32_t* vo,
                      int64_t n, int* temp, const RectGather& rg);

// Super-tiles: SUPER x SUPER tiles of the tile grid.  A gaussian's tile
// rectangle is cut into one reference per super-tile it overlaps; the
// references are sorted by super-tile and each super-tile's references are
// processed in segments of SEG_REFS.
constexpr int SUPER = 16;
constexpr int SEG_REFS = 1024;
inline int super_tiles(int tbx, int tby) {
    return ((tbx + SUPER - 1) / SUPER) * ((tby + SUPER - 1) / SUPER);
}
// Upper bound of the segments of R references over S super-tiles.
inline int64_t segments_bound(int64_t R, int64_t S) { return R / SEG_REFS + S + 1; }
// Super-tiles overlapped by the non-empty tile rectangle [x0, x1) x [y0, y1).
__host__ __device__ inline int super_span(int x0, int y0, int x1, int y1) {
    return ((x1 - 1) / SUPER - x0 / SUPER + 1) * ((y1 - 1) / SUPER - y0 / SUPER + 1);
}

// Binning (binning.hip).  The projection adds the intersection and
// reference totals to the counters above (needed on the host before
// launch_tile_lists); launch_depth_order orders the gaussians by depth,
// gathers their tile rectangles in that order (rect_sorted), with their
// super-tile counts (rcount) and the counts' 1024-block totals (rtot, as
// launch_block_totals leaves them), from which launch_tile_lists' reference
// emission takes each gaussian's first reference slot.
void launch_depth_order(hipStream_t s, int N, uint32_t* dkey, uint32_t* dval, uint32_t* dkey2,
                        uint32_t* dval2, int* radix_temp, int* rank, const uint2* rect, uint2* rect_sorted,
                        int* rcount, int* rtot, const SlotSum* ss, uint32_t** order_out);
// What the depth order still lacks where the totals word says that a key takes
// more than FAR_BITS bits (the same arguments).
void launch_depth_order_far(hipStream_t s, int N, uint32_t* dkey, uint32_t* dval, uint32_t* dkey2,
                            uint32_t* dval2, int* radix_temp, const uint2* rect, uint2* rect_sorted,
                            int* rcount, int* rtot, uint32_t** order_out);

// Scratch of launch_tile_lists for R references, S super-tiles, NS =
// segments_bound(R, S) segments and T tiles.
struct RefBufs {
    uint32_t *key, *val, *key2, *val2;   // R each: references, ping-pong
    int* radix_temp;                     // radix_temp_ints(R)
    int* st_r0;                          // S: reference range of each super-tile;
    int* st_r1;                          //    S; both zero between calls
    int* sstart;                         // S + 1: first segment of each super-tile
    int4* seg;                           // NS: (super-tile, first reference, end reference)
    int* hist;                           // NS * 256: pairs per local tile and segment
    int* tcount;                         // T: pairs per tile
};
// Writes the tile-sorted gaussian ids (I of them) to ids, tile_bins, the
// work items and the summary in meta.
void launch_tile_lists(hipStream_t s, const CamParams& p, int64_t I, int64_t R,
                       const uint32_t* order, const int* rtot,
                       const uint2* rect_sorted, RefBufs rb,
                       uint32_t* ids, int* tscan, int* tile_bins, Items it, TileLists tl,
                       Meta* meta, unsigned long long* isect);
// Ints of the tile scan's scratch (tscan) for T tiles.
inline int64_t tile_scan_ints(int64_t T) { return 3 * ((T + 1023) / 1024) + 8; }

// Raster pair counters: WORK_SLOTS sets of four u64 counters, each set in
// its own 128-byte line (WORK_SLOT_U64 apart); totals are the sums over sets.
constexpr int WORK_SLOTS = 64;
constexpr int WORK_SLOT_U64 = 16;

// Upper bound of the number of (tile, chunk) work items for I intersections.
inline int64_t items_bound(int64_t T, int64_t I) { return T + I / 512 + I / 2048 + 1; }

// Chunks of one tile that a backward record covers: most of a deep tile's
// chunks lie behind every pixel's cutoff and have no work, and a wave of their
// own each, which finds that out after two dependent loads, cost more than the
// chunks that have some (1M gaussians in a blob at 2594x1680: 89k items, 355k
// waves, about 0.2 of 0.62 ms).  Images of few tiles (where every tile is cut
// into chunks) need the chunks' parallelism instead.
inline __host__ __device__ int bwd_group(int64_t T) { return T < 400 ? 1 : 8; }
inline int64_t groups_bound(int64_t T, int64_t I) {
    return bwd_group(T) == 1 ? items_bound(T, I) : T + I / (8 * 512) + 1;
}

// Rasterisation (raster.hip); grids are sized by items_bound / T and the
// kernels read the exact counts from meta.  A non-null `work` (the counter
// sets above) makes the forward add its composited (pixel, entry) pairs to
// counter 0 and its wave-wide entry steps to counter 2, the backward its
// pairs that carry a gradient to counter 1 and its wave-wide entry steps to
// counter 3.
// Training forward: every work item's chunk state (chunked tiles) or final
// pixels (tiles in one piece).  A chunked tile with more than FWD_P chunks
// whose running transmittance is exactly 0 at every pixel after its first
// FWD_P chunks is marked in done[tile] (T ints) and its later chunks, which
// change no output, are not computed; chunked is the tile scan's list.
constexpr int FWD_P = 16;
void launch_raster_fwd(hipStream_t s, const CamParams& p, int64_t max_items, const Meta* meta,
                       Items it, Entries pk, float* final_T, int* final_idx,
                       float* out_img, ChunkBufs cb, unsigned long long* work, const int* chunked,
                       int* done);
// Render-only forward, one workgroup per tile (chunked tiles rasterised chunk
// by chunk up to the merge cutoff); writes the final image, T and index.
void launch_render_tiles(hipStream_t s, const CamParams& p, Items it, Entries pk, float* final_T, int* final_idx, float* out_img,
                         unsigned long long* work);
// Folds the chunked tiles' chunks; live_end[t] (T ints) becomes the item of
// such a tile from which on no pixel has backward work.
void launch_raster_merge(hipStream_t s, const CamParams& p, const Meta* meta, const int* chunked,
                         Items it, float* final_T, int* final_idx, float* out_img, ChunkBufs cb,
                         bool with_suffix, const int* done, int* live_end);
// Fold of the SSIM tiles' loss partials into the loss sum, done by one
// workgroup of a later kernel (the raster backward's first): in float64, in a
// fixed order (thread t adds parts t, t + blockDim.x, ... in order, then a
// tree over the threads), stored to out (which may be coherent host memory
// that the host reads without a stream sync: a system-scope store makes the
// value visible there).  s: 3 x blockDim.x doubles of LDS; blockDim.x a power
// of two.  Every thread of the workgroup calls it.
struct LossFold {
    const float* part;
    int nparts;
    float w;
    float* out;
};
__device__ inline void loss_fold(const LossFold& lf, double* s) {
    const int t = threadIdx.x, nt = blockDim.x;
    double a = 0.0, b = 0.0, n = 0.0;
    for (int i = t; i < lf.nparts; i += nt) {
        a += lf.part[3 * i];
        b += lf.part[3 * i + 1];
        n += lf.part[3 * i + 2];
    }
    s[t] = a;
    s[nt + t] = b;
    s[2 * nt + t] = n;
    __syncthreads();
    for (int off = nt / 2; off > 0; off >>= 1) {
        if (t < off)
            for (int k = 0; k < 3; ++k) s[k * nt + t] += s[k * nt + t + off];
        __syncthreads();
    }
    if (t == 0) {
        const double w = lf.w;
        __hip_atomic_store(lf.out, (float)(w * s[2 * nt] - (w / 3.0) * s[0] + ((1.0 - w) / 3.0) * s[nt]),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __syncthreads();
}
// Workgroup 0 of the launch folds the loss when lf.part is set (loss_fold);
// the items take workgroups 1 ...
void launch_raster_bwd(hipStream_t s, const CamParams& p, int64_t max_groups, const Meta* meta,
                       Items it, Entries pk, const float* final_T,
                       const int* final_idx, ChunkBufs cb, const int* live_end, const float* v_out,
                       float* gacc, unsigned long long* work, const LossFold& lf);
// Adds the six pair counts of the most recent forward/backward into out[6].
void launch_raster_work(hipStream_t s, const CamParams& p, int64_t max_items, const Meta* meta,
                        Items it, Entries pk, const int* final_idx,
                        ChunkBufs cb, const int* live_end, unsigned long long* out);

// The loss: SSIM + L1 forward and backward in tiles whose shape goes by the
// image's size; writes the loss gradient image and one partial (sum SSIM, sum
// L1, pixels) per tile, and returns the number of partials, at most
// ssim_part_bound(H, W).
int ssim_part_bound(int H, int W);
int launch_ssim(hipStream_t s, int H, int W, const float* img, const float* gt, float w,
                float inv_n, float* v_rendered, float* loss_part);



struct AdamHP {
    float step[6];
    float inv_bc2[6];   // 1 / sqrt(1 - beta2^t) per parameter group
    float b1, b2, eps;
};

void launch_sh_rest_adam(hipStream_t s, const CamParams& p, const float4* rec, const int* radii,
                         const float* gacc, float* f_rest, float* m, float* v, const AdamHP& hp);
void launch_proj_bwd_adam(hipStream_t s, const CamParams& p, float* const params[6],
                          float* const m[6], float* const v[6], const AdamHP& hp,
                          GaussOut go, const float* gacc, float* vis, float* gnorm,
                          float* max2d, float inv_max_dim, float* v_mean_out,
                          float* v_scale_out, float* v_quat_out);

// Densification.
struct DensifyHP {
    int N;
    float grad_thresh, size_thresh, screen_thresh;
    int check_screen;
    float cull_alpha, cull_scale, cull_screen;
    int check_huge;
    float half_max_dim;
    int fr;
};
void launch_randn(hipStream_t s, float* dst, int64_t n, uint64_t seed);
void launch_clamp_max(hipStream_t s, float* p, int64_t n, float hi);
// Decides which rows the N gaussians leave (flags: a byte each; tot:
// densify_total_ints(N)) and records the source of each kept row in src (at
// most 3 N); counts_out[0] = rows after the reference's appending,
// counts_out[1] = rows kept.
int64_t densify_total_ints(int64_t N);
void launch_densify(hipStream_t s, const DensifyHP& hp, const float* gnorm, const float* vis,
                    const float* max2d, const float* scales, const float* opac, uint8_t* flags, int* tot,
                    uint2* src, int* counts_out);
// Forms the cnt kept rows of all 18 buffers, one set at a time, in a workspace
// of densify_workspace_floats(cnt, fr) floats and copies them back.
int64_t densify_workspace_floats(int cnt, int fr);
void launch_densify_compact(hipStream_t s, int cnt, int fr, float* const bufs[6], float* const m[6],
                            float* const v[6], const uint2* src, const float* rnd, float* ws);

// Evaluation images: RGBA8 display conversion and PSNR / L1 / SSIM.
struct EvalWindow {
    int ws, pad;      // taps (odd, <= 11) and ws / 2
    float w[11];      // normalised Gaussian taps, computed on the host in fp32
};
int64_t eval_partial_count(int H, int W);
void launch_to_rgba8(hipStream_t s, const float* img, int64_t n, uint32_t* rgba);
void launch_image_metrics(hipStream_t s, const float* img, const float* gt, int H, int W,
                          const EvalWindow& win, double* part, double* out3);

// Nearest-neighbour scales of a point cloud: the points in Morton order and
// a tree of bounding boxes over that order, level after level (level 0: the
// leaves; the last level has one node).
constexpr int KNN_LEVELS = 12;
struct KnnTree {
    int64_t n;
    int levels;
    int64_t cnt[KNN_LEVELS];   // nodes of each level
    int64_t off[KNN_LEVELS];   // first node of each level
    float4* pts;               // n: x, y, z, index bits
    float4* box;               // two per node: low and high corner
};
// Fills n, levels, cnt and off; returns the number of nodes.
int64_t knn_tree_layout(int64_t n, KnnTree& tr);
size_t knn_frame_bytes();
// mean_dist[i] for every point i, unless a coordinate is not finite: word
// (coherent host memory) gets bit 63 and, in its low 32 bits, the first such
// point's index plus one, or 0.  key .. val2: n each.
void launch_knn(hipStream_t s, const float* xyz, const KnnTree& tr, void* frame, uint32_t* key,
                uint32_t* val, uint32_t* key2, uint32_t* val2, int* radix_temp,
                unsigned long long* word, float* mean_dist);

// Target images: area resize and Brown-Conrady undistortion (image.hip).
struct UndistortParams {
    float fx, fy, cx, cy;
    float k1, k2, p1, p2, k3;
    int roi_x, roi_y, roi_w, roi_h;   // crop rectangle of the undistorted image
};
void undistort_roi(int w, int h, UndistortParams& u);   // host: fills roi_*
void launch_resize_area(hipStream_t s, const float* src, int sw, int sh, float* dst, int dw,
                        int dh);
void launch_undistort(hipStream_t s, const float* src, int w, int h, const UndistortParams& u,
                      float* dst);

}  // namespace msp
