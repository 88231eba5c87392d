// knn.hip — initial gaussian scales from the point cloud: for every point the
// mean Euclidean distance to its three nearest other points.
//
// The reference builds a nanoflann kd-tree and asks for the 4 nearest
// neighbours of each point (the point itself first), then averages
// sqrt(d) over neighbours 1..3 (PointsTensor::scales,
// core/include/kdtree_tensor.hpp:26-40; used by Model::Model, model.cpp:63-73).
// Reconstructed clouds are very uneven (dense patches, far outliers), so a
// grid over their bounding box puts thousands of points into one cell.  Here
// the points are sorted along a Morton curve (radix.hip) and a tree of
// bounding boxes is laid over that order: leaves of 16 consecutive points,
// eight children per inner node, levels stored one after the other.  One
// wave answers the 16 queries of one leaf, four lanes per query, each lane
// taking every fourth point of a visited leaf: the walk is the same for the
// whole wave (node numbers and masks live in scalar registers) and visits a
// node while any of its queries may still find a neighbour there.  It starts
// in the queries' own leaf and works up through the siblings of each
// ancestor, so the nearest points along the curve come first and the rest of
// the tree is mostly cut off by the distances already found.
// Squared distances are accumulated per axis like nanoflann's
// L2_Simple_Adaptor ((dx^2 + dy^2) + dz^2 in fp32).  A box's distance is
// formed with the same roundings from per-axis gaps no larger than any of its
// points', so it never exceeds a contained point's distance (rounding is
// monotone) and cutting on it needs no margin: the result is the kd-tree's
// exactly, whatever the order of the points.
// Bound: latency of the dependent node and leaf loads and the vector work of
// the leaf visits (about 40 SIMD cycles per lane and point).  200k points, 60%
// in 40 dense patches and 5% far outliers: 0.265 ms a call (search 183 us,
// sort 64 us, frame 17 us) where the grid search before it took 78 ms, 70 of
// them in the cells of the patches and the rest in a host pass for the
// bounding box.
#include "common.hpp"
#include "kernels.hpp"

namespace msp {

namespace {

constexpr int LEAF = 16;       // points per leaf, queries per wave
constexpr int FAN = 8;         // children per inner node
constexpr int CELLS = 1024;    // Morton cells per axis (10 bits each)

// The cube that the Morton cells divide: the sampled mean of each axis, and
// four times the largest mean absolute deviation to either side (points outside
// take the outermost cells; the boxes come from the points themselves, so the
// cube affects only the order).  Outliers coarsen the cells of the rest less
// than a bounding box does, but both means grow with them: 200k points take 279
// us without, 306 with 1% of them 100 units out, 721 with 1% at 1e4, 726 with
// 0.1% at 1e5 and 10.1 ms with 10% at 1e4 (a grid over the bounding box: 73, 387,
// 73, 73 and 95 ms).  One workgroup, up to 8192 strided samples.
// It also clears the index of the first non-finite point.
struct KnnFrame {
    float lo[3];
    float inv_h;
    unsigned bad;      // first point with a non-finite coordinate, ~0u without any
};

__device__ __forceinline__ double wg_sum(double v, double* sh) {
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += sh[k];
    __syncthreads();
    return t;
}

__global__ __launch_bounds__(1024) void k_knn_frame(int64_t n, const float* __restrict__ xyz,
                                                    KnnFrame* __restrict__ fr) {
    __shared__ double sh[16];
    constexpr int PER = 8;
    const int64_t ns = min(n, (int64_t)1024 * PER);
    float v[PER][3];
    double c = 0.0, m[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int64_t s = (int64_t)j * 1024 + threadIdx.x;
        const int64_t i = s < ns ? s * n / ns : 0;
#pragma unroll
        for (int k = 0; k < 3; ++k) v[j][k] = xyz[3 * i + k];
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        if ((int64_t)j * 1024 + threadIdx.x >= ns) continue;
        c += 1.0;
#pragma unroll
        for (int k = 0; k < 3; ++k) m[k] += (double)v[j][k];
    }
    c = wg_sum(c, sh);
    double dev = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        m[k] = wg_sum(m[k], sh) / c;
        double a = 0.0;
#pragma unroll
        for (int j = 0; j < PER; ++j)
            if ((int64_t)j * 1024 + threadIdx.x < ns) a += fabs((double)v[j][k] - m[k]);
        dev = fmax(dev, wg_sum(a, sh) / c);
    }
    if (threadIdx.x == 0) {
        const double half = 4.0 * dev;
        for (int k = 0; k < 3; ++k) fr->lo[k] = (float)(m[k] - half);
        fr->inv_h = half > 0.0 ? (float)(CELLS / (2.0 * half)) : 0.f;
        fr->bad = ~0u;
    }
}

// Spreads the low 10 bits of v to every third bit.
__device__ __forceinline__ uint32_t spread3(uint32_t v) {
    v = (v | v << 16) & 0x030000FFu;
    v = (v | v << 8) & 0x0300F00Fu;
    v = (v | v << 4) & 0x030C30C3u;
    return (v | v << 2) & 0x09249249u;
}

__device__ __forceinline__ uint32_t cell_of(float v, float lo, float inv_h) {
    // NaN and values outside the cube end up in the outermost cells
    return (uint32_t)(int)fminf(fmaxf((v - lo) * inv_h, 0.f), (float)(CELLS - 1));
}

__global__ __launch_bounds__(256) void k_knn_keys(int64_t n, const float* __restrict__ xyz,
                                                  KnnFrame* __restrict__ fr,
                                                  uint32_t* __restrict__ key,
                                                  uint32_t* __restrict__ val) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float x = xyz[3 * i], y = xyz[3 * i + 1], z = xyz[3 * i + 2];
    if (!(fabsf(x) < INFINITY && fabsf(y) < INFINITY && fabsf(z) < INFINITY))
        atomicMin(&fr->bad, (unsigned)i);
    key[i] = spread3(cell_of(x, fr->lo[0], fr->inv_h)) |
             spread3(cell_of(y, fr->lo[1], fr->inv_h)) << 1 |
             spread3(cell_of(z, fr->lo[2], fr->inv_h)) << 2;
    val[i] = (uint32_t)i;
}

struct Box {
    float lo[3], hi[3];
};

__device__ __forceinline__ Box box_join(const Box& a, const Box& b) {
    Box r;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        r.lo[k] = fminf(a.lo[k], b.lo[k]);
        r.hi[k] = fmaxf(a.hi[k], b.hi[k]);
    }
    return r;
}

__device__ __forceinline__ Box box_load(const float4* __restrict__ box, int64_t node) {
    const float4 a = box[2 * node], b = box[2 * node + 1];
    return Box{{a.x, a.y, a.z}, {b.x, b.y, b.z}};
}

__device__ __forceinline__ void box_store(float4* __restrict__ box, int64_t node, const Box& b) {
    box[2 * node] = make_float4(b.lo[0], b.lo[1], b.lo[2], 0.f);
    box[2 * node + 1] = make_float4(b.hi[0], b.hi[1], b.hi[2], 0.f);
}

// Points in curve order (x, y, z, index bits) and the boxes of levels 0..2: a
// workgroup takes 1024 points, i.e. 64 leaves, 8 nodes of level 1 and one of
// level 2.  Workgroup 0 also publishes the outcome of the finite check (bit
// 63, and the first bad index plus one) for the host.
constexpr int LV_T = LEAF * FAN * FAN;
__global__ __launch_bounds__(LV_T) void k_knn_leaves(KnnTree tr, const float* __restrict__ xyz,
                                                     const uint32_t* __restrict__ order,
                                                     const KnnFrame* __restrict__ fr,
                                                     unsigned long long* word) {
    const int64_t i = (int64_t)blockIdx.x * LV_T + threadIdx.x;
    if (i == 0)
        __hip_atomic_store(word, (1ull << 63) | (unsigned long long)(fr->bad + 1u), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    Box b{{INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}};
    if (i < tr.n) {
        const uint32_t id = order[i];
        const float x = xyz[3 * (size_t)id], y = xyz[3 * (size_t)id + 1], z = xyz[3 * (size_t)id + 2];
        tr.pts[i] = make_float4(x, y, z, __uint_as_float(id));
        b = Box{{x, y, z}, {x, y, z}};
    }
    auto join_lanes = [&](int width) {
        Box o;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            o.lo[k] = __shfl_xor(b.lo[k], width, 64);
            o.hi[k] = __shfl_xor(b.hi[k], width, 64);
        }
        b = box_join(b, o);
    };
    for (int w = 1; w < LEAF; w <<= 1) join_lanes(w);
    const int t = threadIdx.x;
    const int64_t leaf = i / LEAF;
    if (t % LEAF == 0 && leaf < tr.cnt[0]) box_store(tr.box, leaf, b);
    // level 1: eight leaves are 128 points, two waves; the workgroup's 64
    // leaf boxes meet in the first wave through LDS
    __shared__ float s[6][LV_T / LEAF];
    if (t % LEAF == 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            s[k][t / LEAF] = b.lo[k];
            s[3 + k][t / LEAF] = b.hi[k];
        }
    }
    __syncthreads();
    if (t >= LV_T / LEAF) return;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        b.lo[k] = s[k][t];
        b.hi[k] = s[3 + k][t];
    }
    for (int w = 1; w < FAN; w <<= 1) join_lanes(w);
    const int64_t n1 = (int64_t)blockIdx.x * FAN + t / FAN;
    if (t % FAN == 0 && tr.levels > 1 && n1 < tr.cnt[1]) box_store(tr.box, tr.off[1] + n1, b);
    for (int w = FAN; w < FAN * FAN; w <<= 1) join_lanes(w);
    if (t == 0 && tr.levels > 2) box_store(tr.box, tr.off[2] + blockIdx.x, b);
}

// The levels above 2, by one workgroup (a level is an eighth of the one below).
__global__ __launch_bounds__(1024) void k_knn_top(KnnTree tr) {
    for (int l = 3; l < tr.levels; ++l) {
        for (int64_t i = threadIdx.x; i < tr.cnt[l]; i += 1024) {
            Box b = box_load(tr.box, tr.off[l - 1] + FAN * i);
            for (int c = 1; c < FAN && FAN * i + c < tr.cnt[l - 1]; ++c)
                b = box_join(b, box_load(tr.box, tr.off[l - 1] + FAN * i + c));
            box_store(tr.box, tr.off[l] + i, b);
        }
        __syncthreads();
    }
}

// Minimum / maximum over the four lanes of a query.
__device__ __forceinline__ float quad_min(float v) {
    v = fminf(v, dpp<0xB1>(v));
    return fminf(v, dpp<0x4E>(v));
}
__device__ __forceinline__ float quad_max(float v) {
    v = fmaxf(v, dpp<0xB1>(v));
    return fmaxf(v, dpp<0x4E>(v));
}

// The four smallest of this lane's and another lane's ascending four, ascending.
template <int CTRL>
__device__ __forceinline__ void merge4(float* b) {
    float o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = dpp<CTRL>(b[k]);
    float c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) c[k] = fminf(b[k], o[3 - k]);   // bitonic
    const float l0 = fminf(c[0], c[2]), h0 = fmaxf(c[0], c[2]);
    const float l1 = fminf(c[1], c[3]), h1 = fmaxf(c[1], c[3]);
    b[0] = fminf(l0, l1);
    b[1] = fmaxf(l0, l1);
    b[2] = fminf(h0, h1);
    b[3] = fmaxf(h0, h1);
}

__global__ __launch_bounds__(256) void k_knn_search(KnnTree tr, const KnnFrame* __restrict__ fr,
                                                    float* __restrict__ mean_dist) {
    const int leaf0 = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
    if (leaf0 >= tr.cnt[0] || fr->bad != ~0u) return;
    const int lane = threadIdx.x & 63, s = lane & 3;
    const int64_t qi = (int64_t)leaf0 * LEAF + (lane >> 2);
    const float4 q = tr.pts[min(qi, tr.n - 1)];
    // this lane's four smallest squared distances, ascending, and the cut of
    // its query: at least four of the points seen lie within it
    float b[4] = {INFINITY, INFINITY, INFINITY, INFINITY};
    float cut = INFINITY;
    auto visit = [&](int leaf) {
        const int64_t p0 = (int64_t)leaf * LEAF + s;
        float4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = tr.pts[min(p0 + 4 * j, tr.n - 1)];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float dx = q.x - v[j].x, dy = q.y - v[j].y, dz = q.z - v[j].z;
            float d = dx * dx;
            d += dy * dy;
            d += dz * dz;
            if (p0 + 4 * j >= tr.n) d = INFINITY;
            // insertion into the ascending four
            b[3] = __builtin_amdgcn_fmed3f(b[2], b[3], d);
            b[2] = __builtin_amdgcn_fmed3f(b[1], b[2], d);
            b[1] = __builtin_amdgcn_fmed3f(b[0], b[1], d);
            b[0] = fminf(b[0], d);
        }
        // four points lie within a lane's own fourth distance, and one
        // within each lane's first
        cut = fminf(quad_min(b[3]), quad_max(b[0]));
    };
    // Squared distance of this lane's query to node's box.
    auto dist = [&](int64_t node) {
        const Box x = box_load(tr.box, node);
        const float dx = fmaxf(fmaxf(x.lo[0] - q.x, q.x - x.hi[0]), 0.f);
        const float dy = fmaxf(fmaxf(x.lo[1] - q.y, q.y - x.hi[1]), 0.f);
        const float dz = fmaxf(fmaxf(x.lo[2] - q.z, q.z - x.hi[2]), 0.f);
        float d = dx * dx;
        d += dy * dy;
        d += dz * dz;
        return d;
    };
    // Lane s of a query tests children s and s + 4 of a group of eight; its
    // distances are da and db.  Returns the children some query needs.
    float da = 0.f, db = 0.f;
    auto test = [&](int level, int group) {
        const int c0 = group * FAN + s, last = (int)tr.cnt[level] - 1;
        da = dist(tr.off[level] + min(c0, last));
        db = dist(tr.off[level] + min(c0 + 4, last));
        if (c0 > last) da = INFINITY;
        if (c0 + 4 > last) db = INFINITY;
    };
    auto needed = [&]() {
        const uint64_t ma = wave_ballot(da < cut), mb = wave_ballot(db < cut);
        unsigned m = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint64_t lanes = 0x1111111111111111ull << k;
            m |= (ma & lanes ? 1u : 0u) << k | (mb & lanes ? 1u : 0u) << (4 + k);
        }
        return m;
    };
    visit(leaf0);
    int own = leaf0;
    for (int l = 0; l + 1 < tr.levels; ++l, own /= FAN) {
        // the siblings of this level's ancestor, each walked depth first:
        // pend holds the children still to be visited, eight bits a level
        // (at most eight levels lie below the root's children: LEAF FAN^8
        // points are more than an index can hold)
        uint64_t pend = 0;
        int j = l, g = own / FAN;
        test(l, g);
        unsigned m = needed() & ~(1u << (own % FAN));
        for (;;) {
            if (j == 0) {
                // leaves: what is still needed is decided anew after each
                while (m) {
                    const int c = __builtin_ctz(m);
                    m &= ~(1u << c);
                    visit(g * FAN + c);
                    m &= needed();
                }
            }
            if (m) {
                const int c = __builtin_ctz(m);
                pend |= (uint64_t)(m & ~(1u << c)) << (8 * (j - 1));
                g = g * FAN + c;
                --j;
                test(j, g);
                m = needed();
                continue;
            }
            if (j == l) break;
            ++j;
            g /= FAN;
            m = (unsigned)(pend >> (8 * (j - 1))) & 255u;
            pend &= ~(255ull << (8 * (j - 1)));
        }
    }
    merge4<0xB1>(b);
    merge4<0x4E>(b);
    if (s != 0 || qi >= tr.n) return;
    float sum = 0.f;
    sum += sqrtf(b[1]);
    sum += sqrtf(b[2]);
    sum += sqrtf(b[3]);
    mean_dist[__float_as_uint(q.w)] = sum / 3;
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

size_t knn_frame_bytes() { return sizeof(KnnFrame); }

int64_t knn_tree_layout(int64_t n, KnnTree& tr) {
    tr.n = n;
    tr.levels = 0;
    int64_t c = (n + LEAF - 1) / LEAF, off = 0;
    for (;;) {
        tr.cnt[tr.levels] = c;
        tr.off[tr.levels] = off;
        off += c;
        ++tr.levels;
        if (c == 1) break;
        c = (c + FAN - 1) / FAN;
    }
    return off;
}

void launch_knn(hipStream_t s, const float* xyz, const KnnTree& tr, void* frame, uint32_t* key,
                uint32_t* val, uint32_t* key2, uint32_t* val2, int* radix_temp,
                unsigned long long* word, float* mean_dist) {
    KnnFrame* fr = static_cast<KnnFrame*>(frame);
    hipLaunchKernelGGL(k_knn_frame, dim3(1), dim3(1024), 0, s, tr.n, xyz, fr);
    hipLaunchKernelGGL(k_knn_keys, dim3(blocks_for(tr.n)), dim3(256), 0, s, tr.n, xyz, fr, key, val);
    const bool flip = launch_radix_sort(s, key, val, key2, val2, tr.n, 30, radix_temp);
    hipLaunchKernelGGL(k_knn_leaves, dim3((unsigned)((tr.n + LV_T - 1) / LV_T)), dim3(LV_T), 0, s, tr,
                       xyz, (const uint32_t*)(flip ? val2 : val), (const KnnFrame*)fr, word);
    if (tr.levels > 3) hipLaunchKernelGGL(k_knn_top, dim3(1), dim3(1024), 0, s, tr);
    hipLaunchKernelGGL(k_knn_search, dim3((unsigned)((tr.cnt[0] + 3) / 4)), dim3(256), 0, s, tr,
                       (const KnnFrame*)fr, mean_dist);
}

}  // namespace msp
