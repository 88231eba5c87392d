// radix.hip — device-wide scans and a stable LSD radix sort of (u32 key, u32
// value) pairs, used by the binning to order the gaussians by depth and
// their super-tile references by super-tile, and by the nearest-neighbour
// search to order points along a Morton curve.
//
// Sort (more than FUSE_BLOCKS blocks): digits of up to 9 bits,
// reduce-then-scan per pass over 2048-key blocks (512 threads x 4 keys):
//   1. per-block digit histograms in LDS -> hist[digit][block], and the
//      digit totals over all blocks (one global atomic per block and digit)
//   2. one workgroup per digit scans its row of hist and adds the keys of
//      all smaller digits -> scatter offsets
//   3. per-block stable ranks: each wave ranks 256 consecutive keys in
//      four 64-key rounds with a ballot match of equal digits, keeping
//      per-digit running counts in LDS; wave counts are combined in wave
//      order; the block is reordered by digit in LDS and written out in digit
//      runs (coalesced stores).
// Stability makes the result independent of how work is scheduled: equal keys
// keep their input order.
// The depth order sorts with "cull" set: the first pass leaves out the keys
// 0xFFFFFFFF (culled gaussians), and the later passes sort only the visible
// keys (their count, written by the first pass, is read on the device).  The
// last pass writes empty rectangles behind them.
// Depth keys are the bits of the depth less those of the near plane, and the
// depth order sorts their low 27 bits in three passes: depths up to 65536 times
// the near plane.  A fourth (launch_radix_far) follows where the projection
// found a key beyond; the host learns that while the first passes run, and the
// third pass, which a flag on the device tells the same, leaves the rectangles to
// the fourth.  Four passes of 8 bits for all took 13 us more at 500k gaussians, 11
// at 120k.  Renders with some points beyond (or a near plane of 0), with four
// passes of 8 bits / now / the same scene without: 171 / 154 / 136 us for 120k at
// 641x421, 266 / 254 / 236 for 500k and 412 / 398 / 375 for 1.5M at 1297x840, 2187
// / 2150 / 2102 for 6M at 4946x3286 (2230 where the third pass gathered too).
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace msp {

namespace {

constexpr int RT = 512;            // threads per sort block (8 waves)
constexpr int RW = RT / 64;        // waves per sort block
constexpr int RK = 4;              // keys per thread
constexpr int RB = RT * RK;        // keys per block
constexpr int WK = RK * 64;        // keys per wave (RK rounds of 64)
constexpr int SB = SCAN_BLOCK;     // elements per scan block
constexpr int MAX_PASSES = 4;      // 32-bit keys in digits of 8 or 9 bits
constexpr int DBITS = 9;           // bits of the widest digit
constexpr int DMAX = 1 << DBITS;   // its digit slots
constexpr int FUSE_BLOCKS = 64;    // most key blocks of a sort with one kernel a pass
// Groups of equal digits that a wave of depth keys counts with one atomic before
// the rest add one each: a 641x421 render of a wall at one depth (120k gaussians)
// takes 196 us with none and 116 with one; more cost 0.5 us each on spread depths
// and gain nothing.
constexpr int AGG_ROUNDS = 1;
constexpr int DCOPIES = 16;        // copies of the digit totals (block b adds to copy b % 16)

// Digit of key k in a pass: bits [shift, shift + width) (mask).
__device__ __forceinline__ int digit_of(uint32_t k, int shift, uint32_t mask) {
    return (int)((k >> shift) & mask);
}
// Whether a pass with cull leaves key k out.
__device__ __forceinline__ bool culled(uint32_t k, bool cull) { return cull && k == 0xFFFFFFFFu; }

// Keys a pass covers: n, or the count the culling first pass wrote.
__device__ __forceinline__ int64_t pass_n(int64_t n, const int* n_dev) {
    return n_dev ? (int64_t)*n_dev : n;
}

// Sum of v over the NT threads of a block (sh: NT / 64 ints).
template <int NT>
__device__ __forceinline__ int block_sum(int v, int* sh) {
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    int t = 0;
#pragma unroll
    for (int k = 0; k < NT / 64; ++k) t += sh[k];
    __syncthreads();
    return t;
}
__device__ __forceinline__ int block_sum_256(int v, int* sh) { return block_sum<256>(v, sh); }

// Totals of the 1024-element blocks of in.
__global__ __launch_bounds__(256) void k_block_reduce(const int* __restrict__ in, int64_t n,
                                                      int* __restrict__ tot) {
    __shared__ int sh[4];
    const int64_t base = (int64_t)blockIdx.x * SB;
    int v = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int64_t i = base + k * 256 + threadIdx.x;
        if (i < n) v += in[i];
    }
    const int t = block_sum_256(v, sh);
    if (threadIdx.x == 0) tot[blockIdx.x] = t;
}

// Exclusive scan of nb block totals in place (one workgroup); tot[nb] = total.
__global__ __launch_bounds__(1024) void k_scan_totals(int* __restrict__ tot, int nb) {
    __shared__ int s[1024];
    const int per = (nb + 1023) / 1024;
    const int b = min((int)threadIdx.x * per, nb), e = min(b + per, nb);
    int sum = 0;
    for (int i = b; i < e; ++i) sum += tot[i];
    s[threadIdx.x] = sum;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int v = threadIdx.x >= (unsigned)off ? s[threadIdx.x - off] : 0;
        __syncthreads();
        s[threadIdx.x] += v;
        __syncthreads();
    }
    int run = s[threadIdx.x] - sum;
    for (int i = b; i < e; ++i) {
        const int v = tot[i];
        tot[i] = run;
        run += v;
    }
    if (threadIdx.x == 1023) tot[nb] = s[1023];
}

// The SlotSum job, by the first wave of one workgroup: lane k reads slot k's
// counters, the wave sums them and lane 0 publishes the totals word.
__device__ __forceinline__ void slot_sum(const SlotSum& ss) {
    unsigned long long ti = 0, tr = 0, far = 0;
    for (int k = threadIdx.x; k < ISECT_SLOTS; k += 64) {
        ti += __hip_atomic_load(ss.slots + (size_t)k * ISECT_STRIDE, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
        tr += __hip_atomic_load(ss.slots + (size_t)k * ISECT_STRIDE + 1, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
        far |= __hip_atomic_load(ss.slots + (size_t)k * ISECT_STRIDE + 2, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
    }
    const bool any_far = wave_ballot(far != 0) != 0;
    for (int off = 32; off >= 1; off >>= 1) {
        ti += __shfl_xor(ti, off, 64);
        tr += __shfl_xor(tr, off, 64);
    }
    if (threadIdx.x == 0)
        __hip_atomic_store(ss.out, totals_word(ti, tr, any_far), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (ss.far && threadIdx.x == 0) *ss.far = any_far ? 1 : 0;
}

// Super-tiles of a rectangle as the projection packs it, 0 if it is empty.
__device__ __forceinline__ int rect_span(uint2 r) {
    const int x0 = (int)(r.x & 0xFFFFu), y0 = (int)(r.x >> 16);
    const int x1 = (int)(r.y & 0xFFFFu), y1 = (int)(r.y >> 16);
    return (x1 > x0 && y1 > y0) ? super_span(x0, y0, x1, y1) : 0;
}

// Ranks of up to RANK_MAX keys by comparing every key with every other:
// workgroup (x, y) adds to rank[i], for its 256 keys i, the keys of its slice
// of the others that come before (smaller, or equal with a smaller index, so
// the order is a stable sort's).  The other keys are the same for the whole
// workgroup: they come by scalar loads, and a comparison is two vector
// instructions.  rank arrives zeroed (rank_scatter clears it again).  Also
// clears the scan's block totals and does the SlotSum job.
// Few keys leave a radix sort's passes bound by launches, not by work: 12
// launches of 4-6 us for the depth order of 10k gaussians, 66 us, against two
// here, 13 and 4 us.  The comparisons grow with the square of n.  The
// workgroup's own keys go sixteen at a time like the others: one scalar load
// waited for after the other, they made the diagonal workgroups last and the
// launch 18.7 us.
constexpr int RK_T = 256;
__global__ __launch_bounds__(RK_T) void k_rank(const uint32_t* __restrict__ key, int n, int slice,
                                               int* __restrict__ rank, int* __restrict__ tot,
                                               SlotSum ss) {
    if (blockIdx.x == 0 && blockIdx.y == 0) {
        if (ss.out && threadIdx.x < 64) slot_sum(ss);
        if ((int)threadIdx.x < RANK_MAX / SB) tot[threadIdx.x] = 0;
    }
    const int i0 = blockIdx.x * RK_T, i = i0 + threadIdx.x;
    const int j0 = blockIdx.y * slice, j1 = min(j0 + slice, n);
    const uint32_t k = i < n ? key[i] : 0u;
    int c = 0;
    // the slice's keys before this workgroup's, among them, and after them
    const int a = min(max(i0, j0), j1), b = min(max(i0 + RK_T, j0), j1);
    int j = j0;
    for (; j + 16 <= a; j += 16)
#pragma unroll
        for (int u = 0; u < 16; ++u) c += key[j + u] <= k ? 1 : 0;
    for (; j < a; ++j) c += key[j] <= k ? 1 : 0;
    for (; j + 16 <= b; j += 16)
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const uint32_t o = key[j + u];
            c += o < k || (o == k && j + u < i) ? 1 : 0;
        }
    for (; j < b; ++j) {
        const uint32_t o = key[j];
        c += o < k || (o == k && j < i) ? 1 : 0;
    }
    for (; j + 16 <= j1; j += 16)
#pragma unroll
        for (int u = 0; u < 16; ++u) c += key[j + u] < k ? 1 : 0;
    for (; j < j1; ++j) c += key[j] < k ? 1 : 0;
    if (i < n && c) atomicAdd(&rank[i], c);
}

// The ranked values in order, with their rectangles and super-tile counts
// (empty ones for the culled key 0xFFFFFFFF) and the counts' 1024-block totals.
__global__ __launch_bounds__(RK_T) void k_rank_scatter(const uint32_t* __restrict__ key,
                                                       const uint32_t* __restrict__ val, int n,
                                                       int* __restrict__ rank,
                                                       uint32_t* __restrict__ vout,
                                                       int* __restrict__ tot, RectGather rg) {
    __shared__ int s_tot[RANK_MAX / SB];
    const int i = blockIdx.x * RK_T + threadIdx.x;
    if ((int)threadIdx.x < RANK_MAX / SB) s_tot[threadIdx.x] = 0;
    __syncthreads();
    if (i < n) {
        const int r = rank[i];
        rank[i] = 0;
        const uint2 rc = key[i] != 0xFFFFFFFFu ? rg.rect[i] : make_uint2(0u, 0u);
        const int c = rect_span(rc);
        vout[r] = val[i];
        rg.rs[r] = rc;
        rg.cnt[r] = c;
        if (c) atomicAdd(&s_tot[r / SB], c);
    }
    __syncthreads();
    if ((int)threadIdx.x < RANK_MAX / SB && s_tot[threadIdx.x])
        atomicAdd(&tot[threadIdx.x], s_tot[threadIdx.x]);
}

// Per-block digit counts.  D: digit slots (256, or 512 for a 9-bit pass).
// LDS atomics on one address from many lanes of a wave are serialised, so with
// agg (the top bits of depth keys) AGG_ROUNDS groups of equal digits are counted
// with one atomic each.
template <int D>
__global__ __launch_bounds__(RT) void k_radix_hist(const uint32_t* __restrict__ keys, int64_t n,
                                                   const int* __restrict__ n_dev, int shift,
                                                   uint32_t mask, int cull, int agg, int nblocks,
                                                   int* __restrict__ hist, int* __restrict__ dtot,
                                                   SlotSum ss) {
    __shared__ int h[D];
    if (ss.out && blockIdx.x == 0 && threadIdx.x < 64) slot_sum(ss);
    const int64_t ne = pass_n(n, n_dev);
    const int nbe = (int)((ne + RB - 1) / RB);
    if ((int)blockIdx.x >= nbe) return;   // beyond the keys (the offsets scan only the blocks that hold some)
    // this block's key range: the ranges of one XCD's blocks are consecutive
    const int rb = xcd_order((int)blockIdx.x, nbe);
    const int64_t base = (int64_t)rb * RB;
    if (threadIdx.x < D) h[threadIdx.x] = 0;
    __syncthreads();
    const bool cl = cull != 0;
#pragma unroll
    for (int k = 0; k < RK; ++k) {
        const int64_t i = base + k * RT + threadIdx.x;
        const uint32_t key = i < ne ? keys[i] : 0u;
        const int d = digit_of(key, shift, mask);
        bool left = i < ne && !culled(key, cl);
        if (agg) {
            for (int r = 0; r < AGG_ROUNDS; ++r) {
                const uint64_t act = wave_ballot(left);
                if (act == 0) break;
                // the lowest lane still left picks the digit of this round
                const int first = (int)__builtin_ctzll(act);
                const int dl = __builtin_amdgcn_readlane(d, first);
                const uint64_t same = wave_ballot(left && d == dl);
                if ((int)(threadIdx.x & 63) == first) atomicAdd(&h[dl], __popcll(same));
                if (left && d == dl) left = false;
            }
        }
        if (left) atomicAdd(&h[d], 1);
    }
    __syncthreads();
    const int nd = (int)mask + 1;
    if ((int)threadIdx.x < nd) {
        const int c = h[threadIdx.x];
        hist[(size_t)threadIdx.x * nblocks + rb] = c;
        // the digit's total over all blocks, spread over DCOPIES addresses
        if (c) atomicAdd(&dtot[(blockIdx.x % DCOPIES) * D + threadIdx.x], c);
    }
}

// Sorts of at most FUSE_BLOCKS key blocks are launch bound (a kernel here
// takes 4-6 us whatever it does), so they run one kernel a pass: the scatter
// adds up the histograms of all blocks itself, and counts, while it writes
// them out, the digits its keys have in the next pass at the blocks they land
// in.  Histograms are block-major, DMAX digits a row.  k_fused_first counts the
// first pass's digits and clears the later passes' rows.  A 641x421 render with
// three kernels a pass / one: 113 / 102 us for 25k gaussians, 127 / 120 for
// 70k, 139 / 132 for 120k, 154 / 154 for 180k, 169 / 174 for 250k (adding up
// every block's histogram grows with the square of the blocks): the line lies
// at 64 blocks, 131072 keys.
struct FusedPass {
    const int* hist;     // this pass's counts
    int* next;           // the next pass's, or null
    int next_shift;
    uint32_t next_mask;
    int next_agg;        // rounds of equal counts to add up in the wave first
    int* nvis;           // culling pass: gets the number of visible keys
    int* edge0;          // single-pass sort: output range of each digit, or null
    int* edge1;
};
__global__ __launch_bounds__(RT) void k_fused_first(const uint32_t* __restrict__ keys, int n, int shift,
                                                    uint32_t mask, int cull, int* __restrict__ hist,
                                                    int* __restrict__ later, int n_later, int nb,
                                                    SlotSum ss) {
    static_assert(RT == DMAX, "a thread a digit");
    __shared__ int h[DMAX];
    if (ss.out && blockIdx.x == 0 && threadIdx.x < 64) slot_sum(ss);
    const int b = blockIdx.x, tid = threadIdx.x;
    for (int p = 0; p < n_later; ++p) later[((size_t)p * nb + b) * DMAX + tid] = 0;
    h[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RK; ++k) {
        const int i = b * RB + k * RT + tid;
        const uint32_t key = i < n ? keys[i] : 0u;
        if (i < n && !culled(key, cull != 0)) atomicAdd(&h[digit_of(key, shift, mask)], 1);
    }
    __syncthreads();
    hist[(size_t)b * DMAX + tid] = h[tid];
}

// Exclusive scan of one value per thread over the NT threads of a block.
template <int NT>
__device__ __forceinline__ int block_exclusive_scan(int v, int* sh) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) sh[w] = x;
    __syncthreads();
    int wofs = 0;
    for (int k = 0; k < w; ++k) wofs += sh[k];
    __syncthreads();
    return wofs + x - v;
}

// Scatter offsets of one digit (one workgroup per digit d): hist[d][b]
// becomes the position of block b's first key with digit d, i.e. the keys
// of all smaller digits (sum of the dtot copies over d' < d) plus those of
// digit d in the blocks before b (exclusive scan of the row over the blocks
// that hold keys of this pass).
// With edge0 (a single-pass sort) the digit's output range [start, end)
// also goes to edge0[d], edge1[d] when the digit occurs.  With nvis (a culling
// pass) the last digit's workgroup writes its end, the number of visible keys,
// there.
template <int D>
__global__ __launch_bounds__(1024) void k_radix_offsets(int* __restrict__ hist, int nblocks,
                                                        int64_t n, const int* __restrict__ n_dev,
                                                        const int* __restrict__ dtot,
                                                        int* __restrict__ edge0,
                                                        int* __restrict__ edge1,
                                                        int* __restrict__ nvis) {
    __shared__ int sh[16];
    const int d = blockIdx.x, t = threadIdx.x;
    int lower = 0;
    if (t < d) {
#pragma unroll
        for (int c = 0; c < DCOPIES; ++c) lower += dtot[c * D + t];
    }
    int carry = block_sum<1024>(lower, sh);
    const int start = carry;
    const int nbe = (int)((pass_n(n, n_dev) + RB - 1) / RB);
    int* row = hist + (size_t)d * nblocks;
    for (int c = 0; c < nbe; c += 1024) {
        const int i = c + t;
        const int v = i < nbe ? row[i] : 0;
        const int ex = block_exclusive_scan<1024>(v, sh);
        if (i < nbe) row[i] = carry + ex;
        carry += block_sum<1024>(v, sh);
    }
    if (nvis && d == (int)gridDim.x - 1 && t == 0) *nvis = carry;
    if (edge0 && t == 0 && carry > start) {
        edge0[d] = start;
        edge1[d] = carry;
    }
}

// One LSD pass over the digit of each key (digit_of: dbits bits, at most D
// values; with cull the keys 0xFFFFFFFF are left out).  Keys are ranked stably inside the block (each wave ranks its RB/4
// consecutive keys in 64-key rounds by ballot-matching the digit bits and
// keeps per-digit running counts), reordered by digit in LDS, and written out
// in digit runs so that neighbouring lanes store neighbouring addresses.
// With RG (the depth order's last pass) the rectangles of the values go to
// the same positions with their super-tile counts, and the positions past
// the pass's keys (the culled tail) get empty ones.
// FUSED: the offsets come from f.hist and the next pass is counted (FusedPass).
template <bool RG, int D, bool FUSED>
__global__ __launch_bounds__(RT) void k_radix_scatter(const uint32_t* __restrict__ kin,
                                                      const uint32_t* __restrict__ vin,
                                                      uint32_t* __restrict__ kout,
                                                      uint32_t* __restrict__ vout, int64_t n,
                                                      const int* __restrict__ n_dev, int shift,
                                                      uint32_t mask, int cull, int dbits,
                                                      int nblocks, const int* __restrict__ offs,
                                                      int* __restrict__ dtot, RectGather rg, FusedPass f) {
    // The pass's digit totals were last read by the offsets kernel: block 0
    // clears them for the next sort that uses this scratch.
    if (!FUSED && blockIdx.x == 0)
        for (int i = threadIdx.x; i < DCOPIES * D; i += RT) dtot[i] = 0;
    const int64_t ne = pass_n(n, n_dev);
    const int64_t bbase = (int64_t)blockIdx.x * RB;
    const bool gather = RG && !(rg.skip && *rg.skip);
    if (gather) {
        // output positions [ne, n) of this block's range: the culled tail
        for (int64_t p = max(bbase, ne) + threadIdx.x; p < min(bbase + RB, n); p += RT) {
            rg.rs[p] = make_uint2(0u, 0u);
            rg.cnt[p] = 0;
        }
    }
    const int nbe = (int)((ne + RB - 1) / RB);
    if ((int)blockIdx.x >= nbe) return;
    // this block's key range (as in the histogram kernel): the blocks of one
    // XCD write the neighbouring pieces of each digit's output run, which
    // then meet in that XCD's L2 instead of being written back in parts
    const int rb = xcd_order((int)blockIdx.x, nbe);
    const int64_t kbase = (int64_t)rb * RB;
    __shared__ uint32_t s_key[RB];
    __shared__ uint32_t s_val[RB];
    __shared__ int wcnt[RW][D];
    __shared__ int dstart[D];
    __shared__ int gofs[D];
    __shared__ int scan_sh[RW];
    __shared__ int s_nvalid;
    const bool cl = cull != 0;
    const int nd = (int)mask + 1;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    // this block's scatter offset of digit tid, loaded now so that its latency
    // overlaps the key loads and the ranking
    int my_gofs = !FUSED && tid < nd ? offs[(size_t)tid * nblocks + rb] : 0;
    if constexpr (FUSED) {
        // digit tid % D: the keys in all blocks and in those before this one
        // (two threads a digit where there are enough)
        __shared__ int s_half[2][D];
        constexpr int STEP = RT / D;
        const int d = tid % D;
        int total = 0, before = 0;
#pragma unroll 16
        for (int b = tid / D; b < nbe; b += STEP) {
            const int c = f.hist[(size_t)b * DMAX + d];
            total += c;
            before += b < rb ? c : 0;
        }
        if (STEP == 2) {
            if (tid >= D) {
                s_half[0][d] = total;
                s_half[1][d] = before;
            }
            __syncthreads();
            if (tid < D) {
                total += s_half[0][d];
                before += s_half[1][d];
            } else {
                total = 0;
            }
        }
        const int start = block_exclusive_scan<RT>(total, scan_sh);
        my_gofs = start + before;
        if (rb == 0 && tid < nd) {
            if (cl && tid == nd - 1) *f.nvis = start + total;
            if (f.edge0 && total > 0) {
                f.edge0[tid] = start;
                f.edge1[tid] = start + total;
            }
        }
    }
    for (int i = tid; i < RW * D; i += RT) (&wcnt[0][0])[i] = 0;
    __syncthreads();
    const int64_t wbase = kbase + (int64_t)w * WK;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint32_t key[RK], val[RK];
    int dig[RK], rank[RK];
    uint2 rc[RK];      // RG: the value's rectangle, gathered while the keys are ranked
#pragma unroll
    for (int j = 0; j < RK; ++j) {
        const int64_t i = wbase + j * 64 + lane;
        key[j] = i < ne ? kin[i] : 0u;
        val[j] = i < ne ? vin[i] : 0u;
        const bool ok = i < ne && !culled(key[j], cl);
        if (RG) rc[j] = gather && ok ? rg.rect[val[j]] : make_uint2(0u, 0u);
        const int d = ok ? digit_of(key[j], shift, mask) : D;
        dig[j] = d;
        uint64_t peers = wave_ballot(ok);
        if (!ok) peers = ~peers;
        for (int b = 0; b < dbits; ++b) {
            const uint64_t bb = wave_ballot((d >> b) & 1);
            peers &= ((d >> b) & 1) ? bb : ~bb;
        }
        const int before = __popcll(peers & lt);
        const int dd = ok ? d : 0;
        const int base_cnt = ok ? wcnt[w][dd] : 0;
        rank[j] = base_cnt + before;
        // the lowest lane of each digit group advances that digit's count
        if (ok && before == 0) wcnt[w][dd] = base_cnt + __popcll(peers);
    }
    __syncthreads();
    // per digit (threads 0..D-1): offsets of the waves in wave order, the
    // block's count and its start
    int cnt = 0;
    if (tid < D) {
        const int d = tid;
#pragma unroll
        for (int ww = 0; ww < RW; ++ww) {
            const int c = wcnt[ww][d];
            wcnt[ww][d] = cnt;
            cnt += c;
        }
        gofs[d] = my_gofs;
    }
    const int start = block_exclusive_scan<RT>(cnt, scan_sh);
    if (tid < D) dstart[tid] = start;
    if (tid == RT - 1) s_nvalid = start + cnt;
    __syncthreads();
    int lpos[RK];      // each key's place in the block's digit order
#pragma unroll
    for (int j = 0; j < RK; ++j) {
        const int d = dig[j];
        lpos[j] = -1;
        if (d >= D) continue;
        const int p = dstart[d] + wcnt[w][d] + rank[j];
        lpos[j] = p;
        s_key[p] = key[j];
        s_val[p] = val[j];
    }
    __syncthreads();
    const int nvalid = s_nvalid;
    int64_t opos[RK];  // output position of block element tid + u RT
#pragma unroll
    for (int u = 0; u < RK; ++u) {
        const int p = tid + u * RT;
        opos[u] = -1;
        if (p >= nvalid) continue;
        const uint32_t k = s_key[p];
        const int d = digit_of(k, shift, mask);
        const int64_t pos = (int64_t)gofs[d] + (p - dstart[d]);
        kout[pos] = k;
        vout[pos] = s_val[p];
        opos[u] = pos;
        if constexpr (FUSED) {
            if (f.next) {
                const int slot = (int)(pos / RB) * DMAX + digit_of(k, f.next_shift, f.next_mask);
                bool left = true;
                // depth keys: lanes with the same count add once
                for (int r = 0; r < f.next_agg; ++r) {
                    const uint64_t act = wave_ballot(left);
                    if (act == 0) break;
                    const int first = (int)__builtin_ctzll(act);
                    const bool mine = left && slot == __builtin_amdgcn_readlane(slot, first);
                    const uint64_t same = wave_ballot(mine);
                    if (lane == first) atomicAdd(&f.next[slot], __popcll(same));
                    if (mine) left = false;
                }
                if (left) atomicAdd(&f.next[slot], 1);
            }
        }
    }
    if (gather) {
        // the rectangles take the keys' LDS places and go to the same
        // output positions, with their super-tile counts
        __syncthreads();
#pragma unroll
        for (int j = 0; j < RK; ++j) {
            if (lpos[j] < 0) continue;
            s_key[lpos[j]] = rc[j].x;
            s_val[lpos[j]] = rc[j].y;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < RK; ++u) {
            if (opos[u] < 0) continue;
            const int p = tid + u * RT;
            const uint2 r = make_uint2(s_key[p], s_val[p]);
            rg.rs[opos[u]] = r;
            rg.cnt[opos[u]] = rect_span(r);
        }
    }
}

inline unsigned blocks_for(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

int64_t scan_block_count(int64_t n) { return (n + SB - 1) / SB; }

void launch_block_totals(hipStream_t s, const int* in, int64_t n, int* tot) {
    if (n <= 0) return;
    const int nb = (int)scan_block_count(n);
    hipLaunchKernelGGL(k_block_reduce, dim3(nb), dim3(256), 0, s, in, n, tot);
    if (nb > SCAN_DIRECT_BLOCKS) hipLaunchKernelGGL(k_scan_totals, dim3(1), dim3(1024), 0, s, tot, nb);
}

void launch_rank_order(hipStream_t s, const uint32_t* key, const uint32_t* val, int n, int* rank,
                       uint32_t* vout, int* tot, const RectGather& rg, const SlotSum& ss) {
    const int nb = (n + RK_T - 1) / RK_T;
    // about 2048 workgroups, with slices of 64 keys at least
    const int slices = std::max(1, std::min((n + 63) / 64, (2048 + nb - 1) / nb));
    const int slice = ((n + slices - 1) / slices + 15) & ~15;
    hipLaunchKernelGGL(k_rank, dim3(nb, (n + slice - 1) / slice), dim3(RK_T), 0, s, key, n, slice, rank,
                       tot, ss);
    hipLaunchKernelGGL(k_rank_scatter, dim3(nb), dim3(RK_T), 0, s, key, val, n, rank, vout, tot, rg);
}

int64_t radix_temp_ints(int64_t n) {
    const int64_t nb = (n + RB - 1) / RB;
    const int64_t rows = nb <= FUSE_BLOCKS ? nb * MAX_PASSES : nb;
    return DCOPIES * DMAX * MAX_PASSES + rows * DMAX + 16;
}

namespace {

// The three kernels of one pass with D digit slots.
template <int D>
void launch_pass(hipStream_t s, const uint32_t* ki, const uint32_t* vi, uint32_t* ko, uint32_t* vo,
                 int64_t n, const int* n_dev, int shift, uint32_t mask, bool cull, int dbits, bool agg,
                 int nb, int* hist, int* dt, const SlotSum& side, int* edge0, int* edge1, int* nvis,
                 const RectGather* rg) {
    const int nd = (int)mask + 1;
    hipLaunchKernelGGL(k_radix_hist<D>, dim3(nb), dim3(RT), 0, s, ki, n, n_dev, shift, mask,
                       cull ? 1 : 0, agg ? 1 : 0, nb, hist, dt, side);
    hipLaunchKernelGGL(k_radix_offsets<D>, dim3(nd), dim3(1024), 0, s, hist, nb, n, n_dev,
                       (const int*)dt, edge0, edge1, cull ? nvis : nullptr);
    if (rg)
        hipLaunchKernelGGL((k_radix_scatter<true, D, false>), dim3(nb), dim3(RT), 0, s, ki, vi, ko, vo, n,
                           n_dev, shift, mask, cull ? 1 : 0, dbits, nb, (const int*)hist, dt, *rg,
                           FusedPass{});
    else
        hipLaunchKernelGGL((k_radix_scatter<false, D, false>), dim3(nb), dim3(RT), 0, s, ki, vi, ko, vo, n,
                           n_dev, shift, mask, cull ? 1 : 0, dbits, nb, (const int*)hist, dt,
                           RectGather{}, FusedPass{});
}

// One pass of a fused sort (the first pass's counts, then the scatter).
template <int D>
void launch_fused_pass(hipStream_t s, const uint32_t* ki, const uint32_t* vi, uint32_t* ko, uint32_t* vo,
                       int64_t n, const int* n_dev, int shift, uint32_t mask, bool cull, int dbits, int nb,
                       bool first, int* hist, int* later, int n_later, const SlotSum& side, const FusedPass& f,
                       const RectGather* rg) {
    if (first)
        hipLaunchKernelGGL(k_fused_first, dim3(nb), dim3(RT), 0, s, ki, (int)n, shift, mask, cull ? 1 : 0,
                           hist, later, n_later, nb, side);
    if (rg)
        hipLaunchKernelGGL((k_radix_scatter<true, D, true>), dim3(nb), dim3(RT), 0, s, ki, vi, ko, vo, n,
                           n_dev, shift, mask, cull ? 1 : 0, dbits, nb, (const int*)nullptr, (int*)nullptr, *rg,
                           f);
    else
        hipLaunchKernelGGL((k_radix_scatter<false, D, true>), dim3(nb), dim3(RT), 0, s, ki, vi, ko, vo, n,
                           n_dev, shift, mask, cull ? 1 : 0, dbits, nb, (const int*)nullptr, (int*)nullptr,
                           RectGather{}, f);
}

// Scratch layout: the digit totals first, at a fixed place whatever n is
// (DCOPIES x DMAX per pass; each pass's scatter clears its totals for the next
// sort on this scratch), then the per-block histograms (a fused sort has one
// set of rows per pass), then the visible count of a culling sort
// and whether launch_radix_far follows it.
struct RadixTemp {
    int *dtot, *hist, *nvis, *far;
    RadixTemp(int* temp, int nb)
        : dtot(temp), hist(temp + DCOPIES * DMAX * MAX_PASSES),
          nvis(hist + (size_t)DMAX * nb * (nb <= FUSE_BLOCKS ? MAX_PASSES : 1)), far(nvis + 1) {}
};

}  // namespace

// Sorts (k0, v0) by the bits [0, bits) of the keys; ping-pongs with (k1, v1).
// The bits are split into ceil(bits / 9) passes of equal width (fewer digit
// values give longer runs per digit and block).  Returns true when the result
// ends up in (k1, v1).  With rg the last pass also writes each output
// position's rectangle and super-tile count (RectGather); with ss the first
// kernel also does the SlotSum job; with edge0 / edge1 and one pass each
// occurring key value k gets its output range [edge0[k], edge1[k]) (entries of
// absent values are not written).  With cull the keys 0xFFFFFFFF are left out
// by the first pass and the later passes sort only the others; positions
// [visible, n) of the result then hold nothing, and rg marks them empty, unless
// the SlotSum job finds that launch_radix_far has to follow: rg is left to that.
bool launch_radix_sort(hipStream_t s, uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1,
                       int64_t n, int bits, int* temp, const RectGather* rg, const SlotSum* ss,
                       int* edge0, int* edge1, bool cull) {
    if (n <= 0 || bits <= 0) return false;
    const int nb = (int)((n + RB - 1) / RB);
    const int passes = (bits + DBITS - 1) / DBITS;
    const RadixTemp t(temp, nb);
    // the digit totals arrive zeroed: fresh scratch is, and each pass's
    // scatter clears its own
    bool flip = false;
    int shift = 0;
    for (int pass = 0; pass < passes; ++pass) {
        auto width_at = [&](int p, int sh) { return (bits - sh + (passes - p) - 1) / (passes - p); };
        const int width = width_at(pass, shift);
        const uint32_t mask = (1u << width) - 1u;
        const bool pcull = cull && pass == 0, last = pass == passes - 1;
        uint32_t* ki = flip ? k1 : k0;
        uint32_t* vi = flip ? v1 : v0;
        uint32_t* ko = flip ? k0 : k1;
        uint32_t* vo = flip ? v0 : v1;
        const SlotSum side = ss && pass == 0 ? SlotSum{ss->slots, ss->out, t.far} : SlotSum{};
        const int* n_dev = cull && pass > 0 ? t.nvis : nullptr;
        int* e0 = passes == 1 ? edge0 : nullptr;
        int* e1 = passes == 1 ? edge1 : nullptr;
        const RectGather lrg = rg ? RectGather{rg->rect, rg->rs, rg->cnt, ss ? t.far : nullptr} : RectGather{};
        const RectGather* prg = last && rg ? &lrg : nullptr;
        if (nb <= FUSE_BLOCKS) {
            auto rows = [&](int p) { return t.hist + (size_t)p * nb * DMAX; };
            const int nshift = shift + width;
            const FusedPass f{rows(pass), last ? nullptr : rows(pass + 1), nshift,
                              last ? 0u : (1u << width_at(pass + 1, nshift)) - 1u,
                              cull ? AGG_ROUNDS : 0, t.nvis, e0, e1};
            auto go = mask >= 256 ? launch_fused_pass<DMAX> : launch_fused_pass<256>;
            go(s, ki, vi, ko, vo, n, n_dev, shift, mask, pcull, width, nb, pass == 0, rows(0), rows(1),
               passes - 1, side, f, prg);
        } else {
            auto go = mask >= 256 ? launch_pass<DMAX> : launch_pass<256>;
            go(s, ki, vi, ko, vo, n, n_dev, shift, mask, pcull, width, cull && last, nb, t.hist,
               t.dtot + DCOPIES * DMAX * pass, side, e0, e1, t.nvis, prg);
        }
        flip = !flip;
        shift += width;
    }
    return flip;
}

// The pass over the bits from FAR_BITS on, after a culling sort of those below
// on the same scratch.
void launch_radix_far(hipStream_t s, const uint32_t* ki, const uint32_t* vi, uint32_t* ko, uint32_t* vo,
                      int64_t n, int* temp, const RectGather& rg) {
    const int nb = (int)((n + RB - 1) / RB);
    const RadixTemp t(temp, nb);
    constexpr int W = 32 - FAR_BITS;
    launch_pass<256>(s, ki, vi, ko, vo, n, t.nvis, FAR_BITS, (1u << W) - 1u, false, W, true, nb, t.hist,
                     t.dtot + DCOPIES * DMAX * (MAX_PASSES - 1), SlotSum{}, nullptr, nullptr,
                     nullptr, &rg);
}

}  // namespace msp
