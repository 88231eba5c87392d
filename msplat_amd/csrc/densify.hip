// densify.hip — GPU-resident densification: classify, split / duplicate, cull
// and stable compaction of all 18 per-gaussian buffers.
//
// Reference: msplat_densify (msplat_metal.mm:1337-1592) with
// densify_classify_kernel (.metal:3475-3509), densify_append_split_kernel
// (.metal:3514-3600), densify_append_dup_kernel (.metal:3604-3651),
// densify_cull_classify_kernel (.metal:3656-3694), compact_scatter /
// compact_copy_back (.metal:3698-3729) and the two-level block scan
// (.metal:2368-2439).
//
// The reference appends the new rows to every buffer, culls over the 3N-row
// worst case and scatters and copies back each buffer.  Here nothing is
// appended: one pass decides, per gaussian, which of its up to three result
// rows (itself, two children, a duplicate) are kept; a second numbers the kept
// rows (originals, children, duplicates, each in index order, as the
// reference's stable compaction of the appended rows leaves them) and records
// what each is made of; the host reads their count; then, one parameter or
// moment set at a time, a gather forms the rows in a packed workspace and a
// copy brings them back, so that the workspace of a set is still in the
// last-level cache when it is copied.
#include "common.hpp"
#include "kernels.hpp"

namespace msp {

namespace {

__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// Box–Muller from two counter-hashed uniforms per output element.
__global__ __launch_bounds__(256) void k_randn(float* __restrict__ dst, int64_t n, uint64_t seed) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t a = splitmix64(seed ^ (2ull * (uint64_t)i) * 0xD1B54A32D192ED03ull);
    const uint64_t b = splitmix64(a ^ 0x8BB84B93962EACC9ull);
    const float u1 = (float)((a >> 40) + 1) * (1.0f / 16777216.0f);   // (0, 1]
    const float u2 = (float)(b >> 40) * (1.0f / 16777216.0f);         // [0, 1)
    dst[i] = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
}

// What becomes of a gaussian: bits of its flags byte.
constexpr unsigned DF_SPLIT = 1, DF_DUP = 2, DF_KEEP = 4, DF_CHILD = 8, DF_KEEPDUP = 16;
constexpr int DF_T = 256, DF_PER = 4, DF_BLOCK = DF_T * DF_PER;
// Block totals: splits, duplicates, kept originals, kept pairs of children,
// kept duplicates.
constexpr int DF_SUMS = 8;

// Flags of 1024 gaussians per workgroup, and their totals.
__global__ __launch_bounds__(DF_BLOCK) void k_densify_flags(DensifyHP hp, float lsf,
                                                            const float* __restrict__ gnorm,
                                                            const float* __restrict__ vis,
                                                            const float* __restrict__ scales,
                                                            const float* __restrict__ opac,
                                                            const float* __restrict__ max2d,
                                                            uint8_t* __restrict__ flags,
                                                            int* __restrict__ tot) {
    __shared__ int s_n[5];
    if (threadIdx.x < 5) s_n[threadIdx.x] = 0;
    __syncthreads();
    const int i = blockIdx.x * DF_BLOCK + threadIdx.x;
    unsigned f = 0;
    if (i < hp.N) {
        const float s0 = scales[3 * (size_t)i], s1 = scales[3 * (size_t)i + 1], s2 = scales[3 * (size_t)i + 2];
        const float mx = fmaxf(fmaxf(exp_cw(s0), exp_cw(s1)), exp_cw(s2));
        const float vc = vis[i], m2 = max2d[i];
        if (!(vc <= 0.0f)) {
            const float avg = (gnorm[i] / vc) * hp.half_max_dim;
            const bool high = avg > hp.grad_thresh, large = mx > hp.size_thresh;
            if ((large || (hp.check_screen && m2 > hp.screen_thresh)) && high) f |= DF_SPLIT;
            if (!large && high) f |= DF_DUP;
        }
        // the rows' fates: opacity, then size; a split gaussian itself goes,
        // and its children (and a duplicate, which is made after) are
        // smaller by lsf in log scale
        const bool faint = 1.0f / (1.0f + exp_cw(-opac[i])) < hp.cull_alpha;
        const float ms = fmaxf(fmaxf(exp_cw(s0 - lsf), exp_cw(s1 - lsf)), exp_cw(s2 - lsf));
        const bool huge = hp.check_huge && mx > hp.cull_scale;
        const bool huge_small = hp.check_huge && ms > hp.cull_scale;
        const bool on_screen = hp.check_huge && hp.check_screen && m2 > hp.cull_screen;
        if (!faint && !(f & DF_SPLIT) && !huge && !on_screen) f |= DF_KEEP;
        if ((f & DF_SPLIT) && !faint && !huge_small) f |= DF_CHILD;
        if ((f & DF_DUP) && !faint && !((f & DF_SPLIT) ? huge_small : huge)) f |= DF_KEEPDUP;
    }
    if (i < hp.N) flags[i] = (uint8_t)f;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const int n = __popcll(wave_ballot((f >> k) & 1u));
        if ((threadIdx.x & 63) == 0) atomicAdd(&s_n[k], n);
    }
    __syncthreads();
    if (threadIdx.x < 5) tot[DF_SUMS * blockIdx.x + threadIdx.x] = s_n[threadIdx.x];
}

// Source of a result row: the gaussian it comes from, and what it is.
//   0 the gaussian itself, 1 its duplicate, 2 the duplicate of a split one,
//   3 + r its child of random sample r
constexpr unsigned DS_DUP = 1, DS_DUP_SMALL = 2, DS_CHILD = 3;

// Numbers the kept rows.  Workgroup b adds up the totals of all blocks and of
// those before it, scans its own flags, and writes its rows' sources;
// counts_out = (rows the reference would append up to, rows kept).
__global__ __launch_bounds__(DF_T) void k_densify_rows(int N, int nb, const uint8_t* __restrict__ flags,
                                                       const int* __restrict__ tot,
                                                       uint2* __restrict__ src, int* __restrict__ counts_out) {
    __shared__ int s_sum[10];
    __shared__ unsigned long long s_w[DF_T / 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, b = blockIdx.x;
    if (tid < 10) s_sum[tid] = 0;
    __syncthreads();
    int all[5] = {0, 0, 0, 0, 0}, before[5] = {0, 0, 0, 0, 0};
    for (int j = tid; j < nb; j += DF_T)
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const int v = tot[DF_SUMS * j + k];
            all[k] += v;
            before[k] += j < b ? v : 0;
        }
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        for (int off = 32; off >= 1; off >>= 1) {
            all[k] += __shfl_xor(all[k], off, 64);
            before[k] += __shfl_xor(before[k], off, 64);
        }
        if (lane == 0) {
            atomicAdd(&s_sum[k], all[k]);
            atomicAdd(&s_sum[5 + k], before[k]);
        }
    }
    // this thread's four consecutive gaussians; splits, kept originals, kept
    // children pairs and kept duplicates in 16 bits each (a block has 1024)
    const int i0 = b * DF_BLOCK + DF_PER * tid;
    unsigned f[DF_PER];
    unsigned long long c = 0;
#pragma unroll
    for (int u = 0; u < DF_PER; ++u) {
        f[u] = i0 + u < N ? flags[i0 + u] : 0u;
        c += (unsigned long long)(f[u] & 1u) | (unsigned long long)(f[u] >> 2 & 1u) << 16 |
             (unsigned long long)(f[u] >> 3 & 1u) << 32 | (unsigned long long)(f[u] >> 4 & 1u) << 48;
    }
    unsigned long long x = c;
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned long long y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) s_w[w] = x;
    __syncthreads();
    x -= c;
    for (int k = 0; k < w; ++k) x += s_w[k];
    const int kept = s_sum[2], pairs = s_sum[3];
    if (b == 0 && tid == 0) {
        counts_out[0] = N + 2 * s_sum[0] + s_sum[1];
        counts_out[1] = kept + 2 * pairs + s_sum[4];
    }
    int split = s_sum[5] + (int)(x & 0xFFFFu);
    int row = s_sum[7] + (int)(x >> 16 & 0xFFFFu);
    int child = kept + 2 * (s_sum[8] + (int)(x >> 32 & 0xFFFFu));
    int dup = kept + 2 * pairs + s_sum[9] + (int)(x >> 48);
#pragma unroll
    for (int u = 0; u < DF_PER; ++u) {
        const unsigned g = (unsigned)(i0 + u);
        if (f[u] & DF_KEEP) src[row++] = make_uint2(g, 0u);
        if (f[u] & DF_CHILD) {
            src[child++] = make_uint2(g, DS_CHILD + 2 * (unsigned)split);
            src[child++] = make_uint2(g, DS_CHILD + 2 * (unsigned)split + 1);
        }
        if (f[u] & DF_KEEPDUP) src[dup++] = make_uint2(g, f[u] & DF_SPLIT ? DS_DUP_SMALL : DS_DUP);
        if (f[u] & DF_SPLIT) ++split;
    }
}

// Component c of the centre of the child of sample r of the gaussian i: its
// own centre plus the sample, scaled and rotated as the gaussian is.
__device__ __forceinline__ float child_centre(const float* __restrict__ means, const float* __restrict__ scales,
                                              const float* __restrict__ quats, const float* __restrict__ rnd,
                                              size_t i, size_t r, int c) {
    const float* q = quats + 4 * i;
    float qw = q[0], qx = q[1], qy = q[2], qz = q[3];
    const float ql = sqrtf(qw * qw + qx * qx + qy * qy + qz * qz);
    qw /= ql; qx /= ql; qy /= ql; qz /= ql;
    const float r0 = rnd[3 * r] * exp_cw(scales[3 * i]), r1 = rnd[3 * r + 1] * exp_cw(scales[3 * i + 1]),
                r2 = rnd[3 * r + 2] * exp_cw(scales[3 * i + 2]);
    const float v0 = (1 - 2 * (qy * qy + qz * qz)) * r0 + 2 * (qx * qy - qw * qz) * r1 +
                     2 * (qx * qz + qw * qy) * r2;
    const float v1 = 2 * (qx * qy + qw * qz) * r0 + (1 - 2 * (qx * qx + qz * qz)) * r1 +
                     2 * (qy * qz - qw * qx) * r2;
    const float v2 = 2 * (qx * qz - qw * qy) * r0 + 2 * (qy * qz + qw * qx) * r1 +
                     (1 - 2 * (qx * qx + qy * qy)) * r2;
    return means[3 * i + c] + (c == 0 ? v0 : c == 1 ? v1 : v2);
}

// One set of six buffers (parameters, first or second moments) and its place
// in the workspace: buffer k holds cnt rows of st[k] floats at float offset
// off[k] (a multiple of 4).
struct PackedSet {
    float* buf[6];
    int st[6];
    int64_t off[6];
    int64_t f4_end[6];   // cumulative float4 count of the copy-back, buffers 0..k
    int vec[6];          // the buffer is 16-byte aligned (float4 stores)
};

// Gather: workgroup (b, y) takes result rows [256 b, 256 b + 256), of buffer 4
// (features_rest, the widest) for y = 0 and of the others for y = 1.  Rows of
// one workgroup come mostly from consecutive gaussians, so reads coalesce like
// the writes.  PARAMS: children get their own centre, and they and a split
// gaussian's duplicate the smaller scale; otherwise (moments) new rows are zero.
template <bool PARAMS>
__global__ __launch_bounds__(256) void k_gather_rows(PackedSet P, const uint2* __restrict__ src_of,
                                                     int cnt, const float* __restrict__ rnd, float lsf,
                                                     float* __restrict__ ws) {
    __shared__ uint2 s_src[256];
    const int r0 = blockIdx.x * 256, tid = threadIdx.x;
    const int nr = min(256, cnt - r0);
    if (tid < nr) s_src[tid] = src_of[r0 + tid];
    __syncthreads();
    for (int k = 0; k < 6; ++k) {
        const int st = P.st[k];
        if (st == 0 || (k == 4) != (blockIdx.y == 0)) continue;
        const float* __restrict__ src = P.buf[k];
        float* __restrict__ dst = ws + P.off[k] + (int64_t)r0 * st;
        // element e = lr * st + sub, advanced by 256 per step without dividing
        const int q = 256 / st, rem = 256 - q * st;
        int lr = tid / st, sub = tid - lr * st;
        const int ne = nr * st;
        for (int e0 = tid; e0 < ne; e0 += 4 * 256) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                v[u] = 0.f;
                if (e0 + 256 * u < ne) {
                    const uint2 so = s_src[lr];
                    if (PARAMS || so.y == 0u) {
                        v[u] = src[(int64_t)so.x * st + sub];
                        if (PARAMS && k == 0 && so.y >= DS_CHILD)
                            v[u] = child_centre(src, P.buf[1], P.buf[2], rnd, so.x, so.y - DS_CHILD, sub);
                        if (PARAMS && k == 1 && so.y >= DS_DUP_SMALL) v[u] -= lsf;
                    }
                }
                lr += q;
                sub += rem;
                if (sub >= st) { sub -= st; ++lr; }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (e0 + 256 * u < ne) dst[e0 + 256 * u] = v[u];
        }
    }
}

// Copy-back of a set's packed rows: one thread per float4 of the six buffers'
// rows; the workspace regions are 16-byte aligned, a buffer's last float4 may
// be partial, and a buffer that is not 16-byte aligned is copied by scalar
// stores.
__global__ __launch_bounds__(256) void k_copy_back_rows(PackedSet P, int cnt,
                                                        const float* __restrict__ ws) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= P.f4_end[5]) return;
    int k = 0;
    while (t >= P.f4_end[k]) ++k;
    const int64_t i = t - (k ? P.f4_end[k - 1] : 0);
    const int64_t nf = (int64_t)cnt * P.st[k];
    const float* s = ws + P.off[k];
    float* d = P.buf[k];
    if (4 * i + 4 <= nf && P.vec[k]) {
        reinterpret_cast<float4*>(d)[i] = reinterpret_cast<const float4*>(s)[i];
    } else {
        // this thread's own four elements only (fewer at the buffer's end)
        const int64_t e_end = 4 * i + 4 < nf ? 4 * i + 4 : nf;
        for (int64_t e = 4 * i; e < e_end; ++e) d[e] = s[e];
    }
}

// Opacity reset of afterTrain (model.cpp:280-287): logits above hi become hi.
__global__ __launch_bounds__(256) void k_clamp_max(float* __restrict__ p, int64_t n, float hi) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = p[i] > hi ? hi : p[i];
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

void launch_randn(hipStream_t s, float* dst, int64_t n, uint64_t seed) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_randn, dim3(blocks_for(n)), dim3(256), 0, s, dst, n, seed);
}

void launch_clamp_max(hipStream_t s, float* p, int64_t n, float hi) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_clamp_max, dim3(blocks_for(n)), dim3(256), 0, s, p, n, hi);
}

int64_t densify_blocks(int64_t N) { return (N + DF_BLOCK - 1) / DF_BLOCK; }
int64_t densify_total_ints(int64_t N) { return densify_blocks(N) * DF_SUMS; }

void launch_densify(hipStream_t s, const DensifyHP& hp, const float* gnorm, const float* vis,
                    const float* max2d, const float* scales, const float* opac, uint8_t* flags, int* tot,
                    uint2* src, int* counts_out) {
    const int nb = (int)densify_blocks(hp.N);
    hipLaunchKernelGGL(k_densify_flags, dim3(nb), dim3(DF_BLOCK), 0, s, hp, logf(1.6f), gnorm, vis, scales, opac,
                       max2d, flags, tot);
    hipLaunchKernelGGL(k_densify_rows, dim3(nb), dim3(DF_T), 0, s, hp.N, nb, (const uint8_t*)flags,
                       (const int*)tot, src, counts_out);
}

int64_t densify_workspace_floats(int cnt, int fr) {
    const int64_t rows = ((int64_t)cnt + 3) & ~(int64_t)3;
    return rows * (3 + 3 + 4 + 3 + fr + 1);
}

// Per set a gather of about 32 us (52 with the children's centres) and a copy of
// 28 us where 300k SH3 gaussians leave 370k rows, 87 MB a set each way; flags
// and rows take 20 us.  Appending in place, culling 3 N rows and compacting all 18
// buffers at once took 510 us: its workspace, three times as large, no longer
// fitted the last-level cache, and the appending threads wrote whole rows each.
void launch_densify_compact(hipStream_t s, int cnt, int fr, float* const bufs[6], float* const m[6],
                            float* const v[6], const uint2* src, const float* rnd, float* ws) {
    if (cnt <= 0) return;
    const int strides[6] = {3, 3, 4, 3, fr, 1};
    const int64_t cap = ((int64_t)cnt + 3) & ~(int64_t)3;
    float* const* sets[3] = {m, v, bufs};
    for (int set = 0; set < 3; ++set) {
        PackedSet P;
        int64_t off = 0, f4 = 0;
        for (int k = 0; k < 6; ++k) {
            P.buf[k] = sets[set][k];
            P.st[k] = strides[k];
            P.off[k] = off;
            P.vec[k] = (reinterpret_cast<uintptr_t>(P.buf[k]) & 15) == 0;
            off += cap * strides[k];
            f4 += ((int64_t)cnt * strides[k] + 3) / 4;
            P.f4_end[k] = f4;
        }
        const dim3 grid(blocks_for(cnt), 2);
        if (set == 2)
            hipLaunchKernelGGL(k_gather_rows<true>, grid, dim3(256), 0, s, P, src, cnt, rnd, logf(1.6f), ws);
        else
            hipLaunchKernelGGL(k_gather_rows<false>, grid, dim3(256), 0, s, P, src, cnt, rnd, 0.f, ws);
        hipLaunchKernelGGL(k_copy_back_rows, dim3(blocks_for(f4)), dim3(256), 0, s, P, cnt, (const float*)ws);
    }
}

}  // namespace msp
