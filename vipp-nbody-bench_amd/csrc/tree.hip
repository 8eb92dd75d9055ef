// tree.hip - octree build and interaction lists on the GPU.
//
// The reference inserts points one by one into an adaptive octree
// (octree.hpp:79-191).  Its result does not depend on the insertion order:
//  * a point descends by octant o = [x<mid] + 2[y<mid] + 4[z<mid] with
//    mid = (max+min)/2 in FP64 and ties on the high side (first-fit over the
//    children 0..7 with closed bounds, octree.hpp:136,153-158,169-176);
//  * a cell has children iff it holds more than floor(sqrt(8) s) points
//    (octree.hpp:83,143).
// So every point gets a 63-bit path code (3 bits per level, 21 levels) by a
// per-point FP64 midpoint descent, the codes are radix sorted (stable, so equal
// codes keep the caller's order), and the cells of all levels are cut out of the
// sorted codes at once.  Leaves are then sorted by caller index, which is the order
// the reference's leaf vectors have.
#include "gravity.hpp"

#include <algorithm>
#include <cmath>

namespace vg {
namespace {

constexpr double PADDING = 1e-5;  // Problem::OCTREE_WIDTH_PADDING (problem.hpp:167), (double)1E-5L == 1e-5

__global__ __launch_bounds__(256) void k_aabb(const double *__restrict__ x, int64_t n, double *__restrict__ part) {
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    double bad = 0;
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * 256) {
        for (int a = 0; a < 3; ++a) {
            const double v = x[3 * i + a];
            if (!isfinite(v)) bad = 1;
            lo[a] = fmin(lo[a], v);
            hi[a] = fmax(hi[a], v);
        }
    }
    aabb_block_store(lo, hi, bad, part + 7ll * blockIdx.x);
}

// final reduction; box = padded root bounds (fmm.hpp:403-405), box[6] = non-finite flag
__global__ __launch_bounds__(256) void k_aabb_final(const double *__restrict__ part, int nb, double *__restrict__ box) {
    __shared__ double s[7][256];
    double v[7] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY, 0};
    for (int b = threadIdx.x; b < nb; b += 256) {
        for (int a = 0; a < 3; ++a) {
            v[a] = fmin(v[a], part[7 * b + a]);
            v[3 + a] = fmax(v[3 + a], part[7 * b + 3 + a]);
        }
        v[6] = fmax(v[6], part[7 * b + 6]);
    }
    for (int a = 0; a < 7; ++a) s[a][threadIdx.x] = v[a];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < static_cast<unsigned>(w))
            for (int a = 0; a < 7; ++a)
                s[a][threadIdx.x] = a < 3 ? fmin(s[a][threadIdx.x], s[a][threadIdx.x + w]) : fmax(s[a][threadIdx.x], s[a][threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x < 3) {
        box[threadIdx.x] = s[threadIdx.x][0] - PADDING;          // min and max are exact: the order of the reduction does not matter
        box[3 + threadIdx.x] = s[3 + threadIdx.x][0] + PADDING;
    }
    if (threadIdx.x == 0) box[6] = s[6][0];
}

// 63-bit path code: level-1 octant in bits 62..60, level-21 octant in bits 2..0;
// the octants of levels 1..levels only (the bits of deeper levels stay 0: the
// tree reads no digit below the levels it sorts).
__global__ __launch_bounds__(256) void k_codes(const double *__restrict__ x, int64_t n, const double *__restrict__ box, int levels,
                                               uint64_t *__restrict__ key, uint32_t *__restrict__ val) {
    const int64_t i = blockIdx.x * 256ll + threadIdx.x;
    if (i >= n) return;
    double lo[3] = {box[0], box[1], box[2]}, hi[3] = {box[3], box[4], box[5]};
    const double p[3] = {x[3 * i], x[3 * i + 1], x[3 * i + 2]};
    uint64_t code = 0;
    for (int l = 0; l < levels; ++l) {
        unsigned o = 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double mid = (hi[a] + lo[a]) / 2;  // octree.hpp:169
            const bool low = p[a] < mid;
            o |= static_cast<unsigned>(low) << a;
            if (low)
                hi[a] = mid;
            else
                lo[a] = mid;
        }
        code = (code << 3) | o;
    }
    key[i] = code << (3 * (MAXD - levels));
    val[i] = static_cast<uint32_t>(i);
}

// ---- cells of all levels at once ------------------------------------------
// A cell at level d is the run of sorted codes with equal first d octants, and has
// children iff it holds more than thr of them: iff the code thr places after its
// first one still has these d octants.  So each position of the sorted codes tells
// by itself which internal cells start at it: the levels above the octants it shares
// with its predecessor, up to those it shares with the code thr places on.  Counted
// per block and level, scanned, and written in order, level by level, they number
// the internal cells as a level-by-level build would (parents in order, octants in
// order), and internal cell r has the children 1 + 8 r .. 8 + 8 r.
//
// lv[d]: first cell of level d; lv[LV_I + d]: first entry of level d's
// internal cells in int_ids; LV_DEEP: the tree is deeper than the sorted
// octants; LV_NLEAF: non-empty leaves.  Bound by latency and launches: four
// kernels, where a search and a compaction per level took 2 x 11 (100k
// particles), the host's time for a launch each.  Evaluation of 500 particles
// 275 -> 243 us, 16384 492 -> 435, 64000 873 -> 800, 100k 970 -> 878, 4M 9.5 -> 9.45 ms.
constexpr int LV_I = MAXD + 3, LV_DEEP = 2 * (MAXD + 3), LV_NLEAF = LV_DEEP + 1, LV_WORDS = LV_DEEP + 2;

// What the host reads of a build, in pinned memory that the kernels write
// (wait_host_word): two copies and an event are launches of their own, and the
// host has the sizes before the leaves are in order.  RK4 step of 500 particles 654
// -> 596 us, 16384 1.26 -> 1.14 ms, 64,000 2.38 -> 2.27, energies of 256k 1.02 -> 0.97.
// A context's first tree, which no previous one sizes, is read back twice.
struct HostSizes {
    double box[7];
    uint32_t lv[LV_WORDS];
    uint32_t seq;  // number of the build these belong to, written last
};
static_assert(LV_WORDS <= 64, "one wavefront writes the sizes");
__device__ inline void host_sizes(HostSizes *h, uint32_t seq, const double *__restrict__ box, const uint32_t *lv, uint32_t nleaves) {
    if (threadIdx.x >= 64) return;
    if (threadIdx.x < 7) h->box[threadIdx.x] = box[threadIdx.x];
    if (threadIdx.x < LV_WORDS) h->lv[threadIdx.x] = threadIdx.x == LV_NLEAF ? nleaves : lv[threadIdx.x];
    __threadfence_system();
    if (threadIdx.x == 0) __hip_atomic_store(&h->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// cells of the tree in lv, 0 where it has not been built: deeper than the sorted
// octants or more cells than there is room for
__device__ inline int64_t lv_cells(const uint32_t *lv, int SH, int64_t cap) {
    const int64_t nc = 1 + 8ll * lv[LV_I + SH];
    return lv[LV_DEEP] || nc > cap ? 0 : nc;
}
__device__ inline int shared_octants(uint64_t a, uint64_t b) {
    const uint64_t x = a ^ b;
    return x ? (__builtin_clzll(x) - 1) / 3 : MAXD;
}
// Levels 0..SH of the cells of more than thr points that start at position i.
__device__ inline uint32_t cells_at(const uint64_t *__restrict__ key, int64_t n, uint32_t thr, int SH, int64_t i, uint64_t &k) {
    if (i >= n) return 0u;
    k = key[i];
    const uint32_t above = i > 0 ? (2u << shared_octants(key[i - 1], k)) - 1u : 0u;  // levels of which i is not the first code
    const uint32_t upto = i + thr < n ? (2u << min(SH, shared_octants(k, key[i + thr]))) - 1u : 0u;
    return upto & ~above;
}

// cnt[d gridDim.x + b]: cells of level d that start in block b's 256 R positions
__global__ __launch_bounds__(256) void k_cells_count(const uint64_t *__restrict__ key, int64_t n, uint32_t thr, int SH, int R, uint32_t *__restrict__ cnt) {
    __shared__ uint32_t s_cnt[MAXD + 1];
    if (threadIdx.x <= MAXD) s_cnt[threadIdx.x] = 0;
    __syncthreads();
    for (int r = 0; r < R; ++r) {
        uint64_t k;
        for (uint32_t m = cells_at(key, n, thr, SH, (static_cast<int64_t>(blockIdx.x) * R + r) * 256 + threadIdx.x, k); m; m &= m - 1)
            atomicAdd(&s_cnt[__builtin_ctz(m)], 1u);
    }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) <= SH) cnt[static_cast<size_t>(threadIdx.x) * gridDim.x + blockIdx.x] = s_cnt[threadIdx.x];
}

// One block: each level's counts -> exclusive sums over the blocks (a wavefront per
// level), and the level table.
__global__ __launch_bounds__(1024) void k_cells_scan(uint32_t *__restrict__ cnt, int nb, int SH, uint32_t *lv, const double *__restrict__ box,
                                                     HostSizes *host, uint32_t seq) {
    __shared__ uint32_t s_tot[MAXD + 1];
    const int lane = threadIdx.x & 63;
    for (int d = threadIdx.x >> 6; d <= SH; d += 16) {
        uint32_t *row = cnt + static_cast<size_t>(d) * nb;
        uint32_t carry = 0, v = lane < nb ? row[lane] : 0u;
        for (int b0 = 0; b0 < nb; b0 += 64) {
            const int b = b0 + lane;
            const uint32_t nv = b + 64 < nb ? row[b + 64] : 0u;
            uint32_t x = v;
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t y = __shfl_up(x, o, 64);
                if (lane >= o) x += y;
            }
            if (b < nb) row[b] = carry + x - v;
            carry += __shfl(x, 63, 64);
            v = nv;
        }
        if (lane == 0) s_tot[d] = carry;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t at = 0;
        lv[0] = 0;
        for (int d = 0; d <= MAXD + 1; ++d) {
            lv[d + 1] = 1 + 8 * at;
            lv[LV_I + d] = at;
            if (d < SH) at += s_tot[d];
        }
        lv[LV_DEEP] = s_tot[SH] ? 1u : 0u;
        lv[LV_NLEAF] = 0;
    }
    if (!host) return;
    __syncthreads();
    host_sizes(host, seq, box, lv, 0);
}

// The internal cells: id, first position, parent (as an internal cell) and path code, in order.
// A wavefront walks 64 R positions; lane d keeps the number of level d's cells that
// start before the current 64, so a position's rank at each level gives the ids of
// all its ancestors.
__global__ __launch_bounds__(256) void k_cells_write(const uint64_t *__restrict__ key, int64_t n, uint32_t thr, int SH, int R,
                                                     const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ lv, int64_t cap,
                                                     int32_t *__restrict__ int_ids, uint32_t *__restrict__ int_start, int32_t *__restrict__ int_parent,
                                                     uint64_t *__restrict__ int_code) {
    __shared__ uint32_t s_cnt[4][MAXD + 1];
    if (!lv_cells(lv, SH, cap)) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < 4 * (MAXD + 1); i += 256) s_cnt[0][i] = 0;
    __syncthreads();
    const int64_t i0 = (static_cast<int64_t>(blockIdx.x) * 4 + w) * 64 * R + lane;
    uint64_t k = 0;
    for (int r = 0; r < R; ++r)
        for (uint32_t m = cells_at(key, n, thr, SH, i0 + 64 * r, k); m; m &= m - 1) atomicAdd(&s_cnt[w][__builtin_ctz(m)], 1u);
    __syncthreads();
    uint32_t base = 0;
    if (lane < SH) {
        base = lv[LV_I + lane] + cnt[static_cast<size_t>(lane) * gridDim.x + blockIdx.x];
        for (int u = 0; u < w; ++u) base += s_cnt[u][lane];
    }
    for (int r = 0; r < R; ++r) {
        const uint32_t m = cells_at(key, n, thr, SH, i0 + 64 * r, k);
        if (__ballot(m != 0) == 0) continue;
        int32_t id = 0, up = -1;
        for (int d = 0; d < SH; ++d) {
            const uint64_t at = __ballot(m >> d & 1);
            const int32_t rank = static_cast<int32_t>(__builtin_amdgcn_readlane(base, d) + __popcll(at & (~0ull >> (63 - lane)))) - 1;
            if (m >> d & 1) {
                int_ids[rank] = id;
                int_start[rank] = static_cast<uint32_t>(i0 + 64 * r);
                int_parent[rank] = up;
                int_code[rank] = k >> (3 * (MAXD - d));
            }
            up = rank;
            id = 1 + 8 * rank + static_cast<int32_t>(k >> (3 * (MAXD - 1 - d)) & 7u);
            if (lane == d) base += __popcll(at);
        }
    }
}

// The root and the children of the internal cells (octree.hpp:166-191), one per lane.  A child
// ends at the first code, from its parent's first one on, that is past its octant:
// found by doubling steps from thr, then by halving.
__global__ __launch_bounds__(256) void k_cells_expand(const uint64_t *__restrict__ key, int64_t n, uint32_t thr, int SH, uint32_t *lv, int64_t cap,
                                                      const int32_t *__restrict__ int_ids, const uint32_t *__restrict__ int_start,
                                                      const int32_t *__restrict__ int_parent, const double *__restrict__ box, uint32_t *__restrict__ start,
                                                      uint32_t *__restrict__ count, int32_t *__restrict__ child, int32_t *__restrict__ parent,
                                                      uint8_t *__restrict__ octant, int8_t *__restrict__ level, double *__restrict__ bmin,
                                                      double *__restrict__ bmax, int32_t *__restrict__ grid, int32_t *__restrict__ anc,
                                                      uint8_t *__restrict__ flag) {
    const int64_t nc = lv_cells(lv, SH, cap), c = 1 + blockIdx.x * 256ll + threadIdx.x;
    if (c == 1 && nc > 0) {
        start[0] = 0;
        count[0] = static_cast<uint32_t>(n);
        if (n <= thr) child[0] = -1;
        parent[0] = -1;
        octant[0] = 0;
        level[0] = 0;
        flag[0] = n > 0 && n <= thr ? 1 : 0;
        for (int a = 0; a < 3; ++a) {
            // an empty input keeps the zero box of the reference (fmm.hpp:404-405)
            bmin[a] = n ? box[a] : 0.0;
            bmax[a] = n ? box[3 + a] : 0.0;
            grid[a] = 0;
        }
        for (int l = 0; l <= MAXD; ++l) anc[l] = l == 0 ? 0 : -1;
    }
    if (c >= nc) return;
    const int32_t r = static_cast<int32_t>((c - 1) >> 3);
    const unsigned q = threadIdx.x & 7;
    int d = 0;
    while (d + 1 < SH && static_cast<uint32_t>(r) >= lv[LV_I + d + 1]) ++d;
    const int32_t P = int_ids[r];
    const uint32_t s = int_start[r];
    const uint64_t k = key[s];
    const int sh = 3 * (MAXD - 1 - d);
    const uint64_t past = ((k >> (sh + 3)) * 8 + q + 1) << sh;
    int64_t lo = s, hi = s;
    if (k < past) {
        int64_t step = thr;
        hi = lo + step;
        while (hi < n && key[hi] < past) {
            lo = hi;
            step *= 2;
            hi = lo + step;
        }
        if (hi > n) hi = n;
        while (lo + 1 < hi) {
            const int64_t mid = (lo + hi) / 2;
            if (key[mid] < past)
                lo = mid;
            else
                hi = mid;
        }
    }
    const uint32_t end = static_cast<uint32_t>(hi);
    const uint32_t before = __shfl_up(end, 1, 8);
    const uint32_t begin = q == 0 ? s : before, cn = end - begin;
    start[c] = begin;
    count[c] = cn;
    if (cn <= thr) child[c] = -1;  // a child with children gets them from its own lanes
    if (q == 0) child[P] = static_cast<int32_t>(c);
    parent[c] = P;
    octant[c] = static_cast<uint8_t>(q);
    level[c] = static_cast<int8_t>(d + 1);
    flag[c] = cn > 0 && cn <= thr ? 1 : 0;
    double mn[3] = {box[0], box[1], box[2]}, mx[3] = {box[3], box[4], box[5]};
    int32_t g[3] = {0, 0, 0};
    for (int l = 0; l <= d; ++l) {
        const unsigned o = l == d ? q : static_cast<unsigned>(k >> (3 * (MAXD - 1 - l)) & 7u);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double mid = (mx[a] + mn[a]) / 2;  // octree.hpp:169
            const bool low = (o >> a) & 1u;
            mn[a] = low ? mn[a] : mid;
            mx[a] = low ? mid : mx[a];
            g[a] = 2 * g[a] + (low ? 0 : 1);
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        bmin[3 * c + a] = mn[a];
        bmax[3 * c + a] = mx[a];
        grid[3 * c + a] = g[a];
    }
    int32_t *row = anc + c * (MAXD + 1);
    for (int l = MAXD; l > d + 1; --l) row[l] = -1;
    row[d + 1] = static_cast<int32_t>(c);
    for (int32_t l = d, u = r; l >= 0; --l, u = int_parent[u]) row[l] = int_ids[u];
}

// The flagged cells (non-empty leaves) in order, their number into lv: per
// 1024-cell block counts, an exclusive scan of them in one block, then each block
// writes its entries.
__global__ __launch_bounds__(1024) void k_leaf_counts(const uint8_t *__restrict__ flag, const uint32_t *__restrict__ lv, int SH, int64_t cap,
                                                      uint32_t *__restrict__ bcnt) {
    __shared__ uint32_t wsum[16];
    const int64_t i = blockIdx.x * 1024ll + threadIdx.x;
    const uint64_t bal = __ballot(i < lv_cells(lv, SH, cap) && flag[i]);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = __popcll(bal);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int w = 0; w < 16; ++w) t += wsum[w];
        bcnt[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(1024) void k_leaf_scan(uint32_t *__restrict__ bcnt, int nb, uint32_t *lv, const double *__restrict__ box, HostSizes *host, uint32_t seq) {
    __shared__ uint32_t carry;
    __shared__ uint32_t wsum[16];
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    const unsigned lane = threadIdx.x & 63;
    for (int off = 0; off < nb; off += 1024) {
        const int i = off + threadIdx.x;
        const uint32_t v = i < nb ? bcnt[i] : 0u;
        uint32_t x = v;
        for (int s = 1; s < 64; s <<= 1) {
            const uint32_t o = __shfl_up(x, s, 64);
            if (lane >= static_cast<unsigned>(s)) x += o;
        }
        if (lane == 63) wsum[threadIdx.x >> 6] = x;
        __syncthreads();
        uint32_t wb = 0;
        for (unsigned w = 0; w < (threadIdx.x >> 6); ++w) wb += wsum[w];
        const uint32_t c0 = carry;
        if (i < nb) bcnt[i] = c0 + wb + x - v;
        __syncthreads();
        if (threadIdx.x == 1023) carry = c0 + wb + x;
        __syncthreads();
    }
    if (threadIdx.x == 0) lv[LV_NLEAF] = carry;
    host_sizes(host, seq, box, lv, carry);
}

__global__ __launch_bounds__(1024) void k_leaf_write(const uint8_t *__restrict__ flag, const uint32_t *__restrict__ lv, int SH, int64_t cap,
                                                     const uint32_t *__restrict__ boff, int32_t *__restrict__ out) {
    __shared__ uint32_t wsum[16];
    const int64_t i = blockIdx.x * 1024ll + threadIdx.x;
    const unsigned lane = threadIdx.x & 63;
    const bool f = i < lv_cells(lv, SH, cap) && flag[i];
    const uint64_t bal = __ballot(f);
    if (lane == 0) wsum[threadIdx.x >> 6] = __popcll(bal);
    __syncthreads();
    uint32_t wb = boff[blockIdx.x];
    for (unsigned w = 0; w < (threadIdx.x >> 6); ++w) wb += wsum[w];
    if (f) out[wb + __popcll(bal & ((1ull << lane) - 1))] = static_cast<int32_t>(i);
}

// The same in one launch for up to LEAF_BLOCK cells (at most 32 steps of 64 for each
// wavefront; the two launches saved are 7 us of host time): wavefront w of one block takes
// the w-th sixteenth, counts, and writes behind the ones before it.
constexpr int64_t LEAF_BLOCK = 1 << 15;
__global__ __launch_bounds__(1024) void k_leaf_block(const uint8_t *__restrict__ flag, uint32_t *lv, int SH, int64_t cap, int32_t *__restrict__ out,
                                                     const double *__restrict__ box, HostSizes *host, uint32_t seq) {
    __shared__ uint32_t wsum[16];
    const int64_t nc = lv_cells(lv, SH, cap);
    const unsigned lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t per = (nc + 1023) / 1024 * 64, b0 = w * per, b1 = min(nc, b0 + per);
    uint32_t cnt = 0;
    for (int64_t i = b0 + lane; i < b1; i += 64) cnt += flag[i];
    for (int s = 32; s > 0; s >>= 1) cnt += __shfl_xor(cnt, s, 64);
    if (lane == 0) wsum[w] = cnt;
    __syncthreads();
    uint32_t at = 0, all = 0;
    for (unsigned u = 0; u < 16; ++u) {
        if (u < w) at += wsum[u];
        all += wsum[u];
    }
    for (int64_t i = b0; i < b1; i += 64) {
        const bool f = i + lane < b1 && flag[i + lane];
        const uint64_t bal = __ballot(f);
        if (f) out[at + __popcll(bal & ((1ull << lane) - 1))] = static_cast<int32_t>(i + lane);
        at += __popcll(bal);
    }
    if (threadIdx.x == 0) lv[LV_NLEAF] = all;
    host_sizes(host, seq, box, lv, all);
}

// Sort each leaf's caller indices ascending (a leaf holds at most thr points).
__global__ __launch_bounds__(256) void k_leaf_sort(const int32_t *__restrict__ leaves, const uint32_t *__restrict__ start, const uint32_t *__restrict__ count,
                                                   const uint32_t *__restrict__ in, uint32_t *__restrict__ out) {
    extern __shared__ uint32_t sv[];
    const int32_t c = leaves[blockIdx.x];
    const uint32_t s = start[c], n = count[c];
    for (uint32_t i = threadIdx.x; i < n; i += 256) sv[i] = in[s + i];
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += 256) {
        const uint32_t v = sv[i];
        uint32_t r = 0;
        for (uint32_t j = 0; j < n; ++j) r += sv[j] < v;
        out[s + r] = v;
    }
}

// k_leaf_sort with a wavefront per leaf (LS_WAVES leaves per block, LDS of
// LS_WAVES thr words), fused with k_gather: the leaves hold about s points, so
// a block per leaf would leave most of its threads idle.  A lane's first LS_REG points are gathered as soon as their
// caller indices are read, so the random loads of their coordinates overlap
// the ranking; the points of larger leaves beyond 64 LS_REG are gathered after
// it.  Each point is written to its sorted slot with the arithmetic of
// k_gather.
constexpr int LS_WAVES = 4;
constexpr int LS_REG = 3;
constexpr uint32_t LS_MAXTHR = 4096;  // LDS bound of the wavefront form
__global__ __launch_bounds__(64 * LS_WAVES) void k_leaf_sort_w(const int32_t *__restrict__ leaves, const uint32_t *lv,
                                                               const uint32_t *__restrict__ start, const uint32_t *__restrict__ count, uint32_t thr,
                                                               const uint32_t *__restrict__ in, uint32_t *__restrict__ out,
                                                               const double *__restrict__ x, const double *__restrict__ m, double mass,
                                                               const double *__restrict__ box, double eps, double mmax, double *__restrict__ xs64,
                                                               float *__restrict__ xs32) {
    extern __shared__ uint32_t sv[];
    const uint32_t nl = lv[LV_NLEAF];  // 0 when the build did not complete
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t *sw = sv + w * thr;
    const double cx = (box[0] + box[3]) / 2, cy = (box[1] + box[4]) / 2, cz = (box[2] + box[5]) / 2;
    const int ls = length_shift(box, eps);
    const double unit = pow2(-ls), munit = pow2(-mass_shift(ls, mmax, eps));
    auto put = [&](uint32_t k, uint32_t i, double px, double py, double pz, double mi) {
        out[k] = i;
        xs64[4ll * k] = px;
        xs64[4ll * k + 1] = py;
        xs64[4ll * k + 2] = pz;
        xs64[4ll * k + 3] = mi;
        xs32[4ll * k] = static_cast<float>((px - cx) * unit);
        xs32[4ll * k + 1] = static_cast<float>((py - cy) * unit);
        xs32[4ll * k + 2] = static_cast<float>((pz - cz) * unit);
        xs32[4ll * k + 3] = static_cast<float>(mi * munit);
    };
    for (uint32_t j = blockIdx.x * LS_WAVES + w; j < nl; j += gridDim.x * LS_WAVES) {
        const int32_t c = leaves[j];
        const uint32_t s = start[c], n = count[c];
        uint32_t vi[LS_REG];
        double px[LS_REG], py[LS_REG], pz[LS_REG], pm[LS_REG];
#pragma unroll
        for (int u = 0; u < LS_REG; ++u) {
            const uint32_t i = lane + 64u * u;
            vi[u] = i < n ? in[s + i] : 0u;
        }
#pragma unroll
        for (int u = 0; u < LS_REG; ++u) {
            const uint32_t i = lane + 64u * u;
            if (i < n) {
                px[u] = x[3ll * vi[u]];
                py[u] = x[3ll * vi[u] + 1];
                pz[u] = x[3ll * vi[u] + 2];
                pm[u] = m ? m[vi[u]] : mass;
                sw[i] = vi[u];
            }
        }
        for (uint32_t i = lane + 64u * LS_REG; i < n; i += 64) sw[i] = in[s + i];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int u = 0; u < LS_REG; ++u) {
            const uint32_t i = lane + 64u * u;
            if (i < n) {
                uint32_t r = 0;
                for (uint32_t k = 0; k < n; ++k) r += sw[k] < vi[u];
                put(s + r, vi[u], px[u], py[u], pz[u], pm[u]);
            }
        }
        for (uint32_t i = lane + 64u * LS_REG; i < n; i += 64) {
            const uint32_t v = sw[i];
            uint32_t r = 0;
            for (uint32_t k = 0; k < n; ++k) r += sw[k] < v;
            put(s + r, v, x[3ll * v], x[3ll * v + 1], x[3ll * v + 2], m ? m[v] : mass);
        }
        __builtin_amdgcn_wave_barrier();  // every lane has read sw before the next leaf overwrites it
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

__global__ __launch_bounds__(256) void k_gather(const uint32_t *__restrict__ perm, int64_t n, const double *__restrict__ x, const double *__restrict__ m,
                                                double mass, const double *__restrict__ box, double eps, double mmax, double *__restrict__ xs64,
                                                float *__restrict__ xs32) {
    const int64_t k = blockIdx.x * 256ll + threadIdx.x;
    if (k >= n) return;
    const uint32_t i = perm[k];
    const double px = x[3ll * i], py = x[3ll * i + 1], pz = x[3ll * i + 2];
    const double mi = m ? m[i] : mass;
    xs64[4 * k] = px;
    xs64[4 * k + 1] = py;
    xs64[4 * k + 2] = pz;
    xs64[4 * k + 3] = mi;
    const double cx = (box[0] + box[3]) / 2, cy = (box[1] + box[4]) / 2, cz = (box[2] + box[5]) / 2;
    const int ls = length_shift(box, eps);
    const double unit = pow2(-ls), munit = pow2(-mass_shift(ls, mmax, eps));
    xs32[4 * k] = static_cast<float>((px - cx) * unit);
    xs32[4 * k + 1] = static_cast<float>((py - cy) * unit);
    xs32[4 * k + 2] = static_cast<float>((pz - cz) * unit);
    xs32[4 * k + 3] = static_cast<float>(mi * munit);
}

// ---------------------------------------------------------------------------
// Interaction lists of all levels at once (calc_link, solver_ref.hpp:115-162)
// ---------------------------------------------------------------------------
// The NB list of an internal cell holds the internal cells of its level that
// touch it or are itself: the parents of two such cells touch as well, and are
// internal.  calc_link takes candidates in the order of the parent's NB list and
// of their octants, and the root's list is the root, so every NB list is in the order
// of the path codes.  So a cell's NB list needs no list of its parent: its 27
// neighbour positions are looked up among its level's internal cells, which are in
// the order of their path codes.  Bound by latency (a wavefront per cell: the
// search's 5 to 17 dependent reads, then one of the candidates); one launch for
// all levels, where a launch per level waited for the one before (and 64 candidates'
// positions, read from memory, are now their octant and place): 500 particles 22 -> 10 us,
// 1M at s = 64 56 to 107 -> 20.  Evaluation of 500 particles 191 -> 180 us, 16384 413 -> 380,
// 64000 767 -> 729, 1M clustered 2.67 -> 2.55 ms.
__device__ inline uint64_t spread3(uint32_t x) {  // bit i of 21 to bit 3 i
    uint64_t v = x & 0x1fffffu;
    v = (v | v << 32) & 0x1f00000000ffffull;
    v = (v | v << 16) & 0x1f0000ff0000ffull;
    v = (v | v << 8) & 0x100f00f00f00f00full;
    v = (v | v << 4) & 0x10c30c30c30c30c3ull;
    v = (v | v << 2) & 0x1249249249249249ull;
    return v;
}
// Path code of a position at level d (octant bit a is set on the low side, octree.hpp:164-176).
__device__ inline uint64_t path_code(int d, int x, int y, int z) {
    const uint32_t m = (1u << d) - 1;
    return spread3(~static_cast<uint32_t>(x) & m) | spread3(~static_cast<uint32_t>(y) & m) << 1 | spread3(~static_cast<uint32_t>(z) & m) << 2;
}

// NB list of one internal cell and the NI and AP lists of its 8 children per wavefront
// (4 per block), and the number of particles in the NI cells of each (the P2P's sources).
// The children share their candidates: the children of the
// cell's NB cells, taken in the order of solver_ref.hpp:129-147 (NB entry e, child
// offset q).  Lane l tests candidate 64 r + l of round r against all 8
// siblings; each sibling's NI / AP entries are appended in candidate
// order through ballots and prefix popcounts, so the lists come out in the
// reference's order.  An entry needs no bound check: a cell has 27 positions
// around it, and 8 x 27 candidates of which its 27 are not AP.
__global__ __launch_bounds__(256) void k_lists(const uint32_t *__restrict__ lv, int SH, int64_t cap, const int32_t *__restrict__ int_ids,
                                               const uint64_t *__restrict__ int_code, const int8_t *__restrict__ level, const int32_t *__restrict__ child,
                                               const int32_t *__restrict__ grid, int32_t *__restrict__ nb, int32_t *__restrict__ ni, int32_t *__restrict__ ap,
                                               int32_t *__restrict__ nb_cnt, int32_t *__restrict__ ni_cnt, int32_t *__restrict__ ap_cnt,
                                               int32_t *__restrict__ nbr27, const uint32_t *__restrict__ count, uint32_t *__restrict__ local) {
    __shared__ int32_t s_r[4][28], s_o[4][28];
    const int64_t nc = lv_cells(lv, SH, cap), nint = nc / 8;  // nc = 1 + 8 nint
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (blockIdx.x == 0 && threadIdx.x == 0 && nc > 0) {  // the root (solver_ref.hpp:149-152); with children, its NB list is its own wavefront's
        ap_cnt[0] = 0;
        ni_cnt[0] = nint ? 0 : 1;
        local[0] = nint ? 0 : count[0];
        if (nint == 0) {
            ni[0] = 0;
            nb_cnt[0] = 0;
        }
    }
    const int64_t r = blockIdx.x * 4ll + w;
    if (r >= nint) return;  // whole wavefront
    const int32_t P = int_ids[r], cb = static_cast<int32_t>(1 + 8 * r);
    const int d = level[P];
    const int px = grid[3 * P], py = grid[3 * P + 1], pz = grid[3 * P + 2];
    bool leaf[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) leaf[t] = child[cb + t] < 0;
    // lane l < 27: the internal cell at offset (l % 3 - 1, l / 3 % 3 - 1, l / 9 - 1), as an entry of int_ids, or -1
    int32_t found = -1;
    {
        const int x = px + lane % 3 - 1, y = py + lane / 3 % 3 - 1, z = pz + lane / 9 - 1, side = 1 << d;
        if (lane < 27 && x >= 0 && x < side && y >= 0 && y < side && z >= 0 && z < side) {
            const uint64_t code = path_code(d, x, y, z);
            uint32_t lo = lv[LV_I + d], hi = lv[LV_I + d + 1];  // the last cell whose code is not above
            while (lo + 1 < hi) {
                const uint32_t mid = (lo + hi) / 2;
                if (int_code[mid] <= code)
                    lo = mid;
                else
                    hi = mid;
            }
            if (int_code[lo] == code) found = static_cast<int32_t>(lo);
        }
    }
    int at = 0;  // its place in the NB list
    const int npn = __popcll(__ballot(found >= 0));
    for (int l = 0; l < 27; ++l) {
        const int32_t o = __builtin_amdgcn_readlane(found, l);
        at += o >= 0 && o < found;
    }
    if (lane < 27) {
        int32_t id = -1;
        if (found >= 0) {
            id = int_ids[found];
            s_r[w][at] = found;
            s_o[w][at] = lane;
            nb[27 * static_cast<int64_t>(P) + at] = id;
        }
        nbr27[27 * static_cast<int64_t>(P) + lane] = id;
    }
    if (lane == 0) nb_cnt[P] = npn;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint64_t below = (1ull << lane) - 1;
    int nin[8], apn[8];
    uint32_t src[8];  // this lane's share of the particles in each child's NI cells
#pragma unroll
    for (int t = 0; t < 8; ++t) nin[t] = apn[t] = 0, src[t] = 0;
    const int ncand = 8 * npn;
    for (int r0 = 0; r0 < ncand; r0 += 64) {
        const int cand = r0 + lane, q = lane & 7;
        const bool valid = cand < ncand;
        int32_t cc = 0;
        int cx = 0, cy = 0, cz = 0;  // position relative to the first child position of P
        bool cint = false;
        uint32_t cn = 0;
        if (valid) {
            const int o = s_o[w][cand / 8];
            cc = 1 + 8 * s_r[w][cand / 8] + q;
            cx = 2 * (o % 3 - 1) + 1 - (q & 1);
            cy = 2 * (o / 3 % 3 - 1) + 1 - (q >> 1 & 1);
            cz = 2 * (o / 9 - 1) + 1 - (q >> 2);
            cint = child[cc] >= 0;
            cn = count[cc];
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int32_t ct = cb + t;
            const int dx = cx - (1 - (t & 1)), dy = cy - (1 - (t >> 1 & 1)), dz = cz - (1 - (t >> 2));
            const bool adj = dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1 && dz >= -1 && dz <= 1;  // fmm.hpp:475-493
            const bool isni = valid && adj && (leaf[t] || !cint);
            const bool isap = valid && !adj;
            const uint64_t mni = __ballot(isni), map = __ballot(isap);
            if (isni) ni[27 * static_cast<int64_t>(ct) + nin[t] + __popcll(mni & below)] = cc;
            if (isap) ap[189 * static_cast<int64_t>(ct) + apn[t] + __popcll(map & below)] = cc;
            nin[t] += __popcll(mni);
            apn[t] += __popcll(map);
            src[t] += isni ? cn : 0u;
        }
    }
#pragma unroll
    for (int t = 0; t < 8; ++t)
        for (int s = 32; s > 0; s >>= 1) src[t] += __shfl_xor(src[t], s, 64);
    if (lane < 8) {
        int b = 0, e = 0;
        uint32_t n = 0;
        bool lf = false;
#pragma unroll
        for (int t = 0; t < 8; ++t)
            if (lane == t) b = nin[t], e = apn[t], n = src[t], lf = leaf[t];
        if (lf) nb_cnt[cb + lane] = 0;  // an internal child has its own wavefront
        ni_cnt[cb + lane] = b;
        ap_cnt[cb + lane] = e;
        local[cb + lane] = n;
    }
}

// ---------------------------------------------------------------------------
// Reference numbering (for export): children of the internal cell that
// subdivided r-th are 1 + 8r .. 8 + 8r (octree.hpp:170-177).  A cell
// subdivides when its (thr+1)-th point in caller order arrives; cells that
// subdivide on the same arrival do so parent first.  So internal cells are
// ranked by (t = (thr+1)-th smallest caller index of the cell, depth).
// S(cell) = its thr+1 smallest caller indices, merged bottom-up.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_smallest(const int32_t *__restrict__ ids, int n_ids, const int32_t *__restrict__ child, const uint32_t *__restrict__ start,
                                                  const uint32_t *__restrict__ count, const uint32_t *__restrict__ perm, const int32_t *__restrict__ int_index,
                                                  uint32_t *__restrict__ slist, uint32_t keep, uint64_t *__restrict__ rkey, uint32_t *__restrict__ rval,
                                                  const int8_t *__restrict__ level, int pow2) {
    extern __shared__ uint32_t buf[];
    const int32_t P = ids[blockIdx.x];
    const int32_t base = child[P];
    // gather candidates
    __shared__ uint32_t off[9];
    if (threadIdx.x == 0) {
        uint32_t o = 0;
        for (int q = 0; q < 8; ++q) {
            off[q] = o;
            const int32_t c = base + q;
            o += child[c] < 0 ? count[c] : keep;
        }
        off[8] = o;
    }
    __syncthreads();
    for (int q = 0; q < 8; ++q) {
        const int32_t c = base + q;
        const uint32_t n = off[q + 1] - off[q];
        const uint32_t *src = child[c] < 0 ? perm + start[c] : slist + static_cast<size_t>(int_index[c]) * keep;
        for (uint32_t i = threadIdx.x; i < n; i += 256) buf[off[q] + i] = src[i];
    }
    for (uint32_t i = off[8] + threadIdx.x; i < static_cast<uint32_t>(pow2); i += 256) buf[i] = 0xFFFFFFFFu;
    __syncthreads();
    // bitonic sort of pow2 entries
    for (int k = 2; k <= pow2; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = threadIdx.x; i < pow2; i += 256) {
                const int l = i ^ j;
                if (l > i) {
                    const uint32_t a = buf[i], b = buf[l];
                    const bool up = (i & k) == 0;
                    if ((a > b) == up) {
                        buf[i] = b;
                        buf[l] = a;
                    }
                }
            }
            __syncthreads();
        }
    }
    const int32_t me = int_index[P];
    for (uint32_t i = threadIdx.x; i < keep; i += 256) slist[static_cast<size_t>(me) * keep + i] = buf[i];
    if (threadIdx.x == 0) {
        rkey[me] = (static_cast<uint64_t>(buf[keep - 1]) << 5) | static_cast<uint64_t>(level[P]);
        rval[me] = static_cast<uint32_t>(me);
    }
}

__global__ __launch_bounds__(256) void k_int_index(const int32_t *__restrict__ int_ids, int64_t nint, int32_t *__restrict__ int_index) {
    const int64_t k = blockIdx.x * 256ll + threadIdx.x;
    if (k < nint) int_index[int_ids[k]] = static_cast<int32_t>(k);
}

__global__ __launch_bounds__(256) void k_rank_of(const uint32_t *__restrict__ sorted_val, int64_t nint, int32_t *__restrict__ rank) {
    const int64_t r = blockIdx.x * 256ll + threadIdx.x;
    if (r < nint) rank[sorted_val[r]] = static_cast<int32_t>(r);
}

__global__ __launch_bounds__(256) void k_ref_ids(int64_t nc, const int32_t *__restrict__ parent, const uint8_t *__restrict__ octant,
                                                 const int32_t *__restrict__ int_index, const int32_t *__restrict__ rank, int32_t *__restrict__ ref_id) {
    const int64_t c = blockIdx.x * 256ll + threadIdx.x;
    if (c >= nc) return;
    const int32_t P = parent[c];
    ref_id[c] = P < 0 ? 0 : 1 + 8 * rank[int_index[P]] + octant[c];
}

}  // namespace

static void ensure_cells(TreeDev &t, int64_t ncell) {
    t.start.ensure(ncell);
    t.count.ensure(ncell);
    t.child.ensure(ncell);
    t.parent.ensure(ncell);
    t.octant.ensure(ncell);
    t.level.ensure(ncell);
    t.bmin.ensure(3 * ncell);
    t.bmax.ensure(3 * ncell);
    t.grid.ensure(3 * ncell);
    t.anc.ensure((MAXD + 1) * ncell);
    t.flags.ensure(ncell);
    t.leaf_ids.ensure(ncell);
    t.int_ids.ensure(ncell / 8 + 1);
    t.int_start.ensure(ncell / 8 + 1);
    t.int_parent.ensure(ncell / 8 + 1);
    t.int_code.ensure(ncell / 8 + 1);
}

// The lists of a tree of at most cap cells, whose sizes the level table holds.
static void lists_enqueue(Ctx &c, int SH, int64_t cap) {
    TreeDev &t = c.t;
    t.nb.ensure(27 * cap);
    t.ni.ensure(27 * cap);
    t.ap.ensure(189 * cap);
    t.nb_cnt.ensure(cap);
    t.ni_cnt.ensure(cap);
    t.ap_cnt.ensure(cap);
    t.nbr27.ensure(27 * cap);
    c.p2p_local.ensure(cap);
    k_lists<<<ceil_div(std::max<int64_t>(1, cap / 8), 4), 256, 0, c.stream>>>(t.lv, SH, cap, t.int_ids, t.int_code, t.level, t.child, t.grid, t.nb, t.ni,
                                                                            t.ap, t.nb_cnt, t.ni_cnt, t.ap_cnt, t.nbr27, t.count, c.p2p_local);
    VG_LAUNCH_CHECK();
}

// With ahead, the operators (which need the root box alone) and the lists of trees of
// up to AHEAD_CELLS cells (room for the lists of twice the last tree's cells: at most
// 283 MB) are enqueued behind the tree before the host waits for its sizes: the
// device forms them while the host wakes up.
constexpr int64_t AHEAD_CELLS = 1 << 18;
void tree_build(Ctx &c, bool ahead) {
    hipStream_t st = c.stream;
    TreeDev &t = c.t;
    const int64_t n = c.n;
    // 1. root box
    //    (the RK4 stage that wrote x may have left its partial boxes)
    c.box.ensure(8);
    if (c.aabb_parts > 0) {
        k_aabb_final<<<1, 256, 0, st>>>(c.aabb_part, c.aabb_parts, c.box);
    } else {
        const int nb = static_cast<int>(std::min<int64_t>(1024, std::max<int64_t>(1, (n + 255) / 256)));
        c.aabb_part.ensure(7 * static_cast<size_t>(nb));
        k_aabb<<<nb, 256, 0, st>>>(c.x, n, c.aabb_part);
        k_aabb_final<<<1, 256, 0, st>>>(c.aabb_part, nb, c.box);
    }
    c.aabb_parts = 0;
    VG_LAUNCH_CHECK();
    const int64_t n1 = std::max<int64_t>(1, n);
    for (int b = 0; b < 2; ++b) {
        c.key[b].ensure(n1);
        c.val[b].ensure(n1);
    }
    c.perm.ensure(n1);
    c.xs64.ensure(4 * n1);
    c.xs32.ensure(4 * n1);
    t.lv.ensure(LV_WORDS);
    uint64_t *k0 = c.key[0].p, *k1 = c.key[1].p;
    uint32_t *v0 = c.val[0].p, *v1 = c.val[1].p;
    HostSizes *host = reinterpret_cast<HostSizes *>(static_cast<char *>(c.pinned) + 512);
    static_assert(512 + sizeof(HostSizes) <= Ctx::PINNED_BYTES, "pinned words");
    const uint32_t *hlv = host->lv;
    // 2. path codes and a stable sort of the octants of levels 1..SH (bits below
    //    the deepest level do not matter: leaves are re-sorted by caller index): two
    //    levels beyond the previous tree's depth (consecutive evaluations differ
    //    little), 16 for the first tree (a first step of 500 particles takes 1.24 ms, a
    //    later one 0.6); a tree that needs a deeper level is built
    //    again with all 21 sorted.
    int SH = t.depth > 0 ? std::min(MAXD, t.depth + 2) : 16;
    const int R = n <= (1 << 20) ? 4 : 16;  // positions per lane: blocks for every CU, then fewer counts to scan
    const int nb = static_cast<int>(ceil_div(n, 256 * R));
    c.cmp_cnt.ensure(std::max<int64_t>(1, static_cast<int64_t>(nb) * (MAXD + 1)));
    // 3. room for twice the previous tree's cells; the first tree's are counted first
    int64_t cap = t.ncells > 0 ? std::max<int64_t>(1024, 2 * t.ncells) : 0;
    ensure_cells(t, std::max<int64_t>(1, cap));
    auto sort_and_count = [&] {
        if (n) {
            k_codes<<<ceil_div(n, 256), 256, 0, st>>>(c.x, n, c.box, SH, k0, v0);
            if (n > c.thr) radix_sort_pairs(st, k0, v0, k1, v1, n, 3 * (MAXD - SH), 3 * MAXD, c.rs_hist);
            k_cells_count<<<nb, 256, 0, st>>>(k0, n, c.thr, SH, R, c.cmp_cnt);
        }
        k_cells_scan<<<1, 1024, 0, st>>>(c.cmp_cnt, nb, SH, t.lv, c.box, cap > 0 ? nullptr : host, c.tree_seq);
        VG_LAUNCH_CHECK();
    };
    // 4. cells, the non-empty leaves, leaf order by caller index, particles in sorted order
    auto cells = [&] {
        if (n > c.thr) k_cells_write<<<nb, 256, 0, st>>>(k0, n, c.thr, SH, R, c.cmp_cnt, t.lv, cap, t.int_ids, t.int_start, t.int_parent, t.int_code);
        k_cells_expand<<<ceil_div(cap, 256), 256, 0, st>>>(k0, n, c.thr, SH, t.lv, cap, t.int_ids, t.int_start, t.int_parent, c.box, t.start, t.count, t.child,
                                                           t.parent, t.octant, t.level, t.bmin, t.bmax, t.grid, t.anc, t.flags);
        if (cap <= LEAF_BLOCK) {
            k_leaf_block<<<1, 1024, 0, st>>>(t.flags, t.lv, SH, cap, t.leaf_ids, c.box, host, c.tree_seq);
        } else {
            const unsigned gl = ceil_div(cap, 1024);
            t.leaf_cnt.ensure(gl);
            k_leaf_counts<<<gl, 1024, 0, st>>>(t.flags, t.lv, SH, cap, t.leaf_cnt);
            k_leaf_scan<<<1, 1024, 0, st>>>(t.leaf_cnt, static_cast<int>(gl), t.lv, c.box, host, c.tree_seq);
            k_leaf_write<<<gl, 1024, 0, st>>>(t.flags, t.lv, SH, cap, t.leaf_cnt, t.leaf_ids);
        }
        if (n && c.thr <= LS_MAXTHR) {
            // a wavefront per leaf of the previous tree and a quarter more (the leaf
            // count changes little; the blocks loop over any excess)
            const int64_t leaves = t.nleaves > 0 ? std::max<int64_t>(1024, t.nleaves + t.nleaves / 4) : cap;
            k_leaf_sort_w<<<ceil_div(std::min(cap, leaves), LS_WAVES), 64 * LS_WAVES, LS_WAVES * c.thr * sizeof(uint32_t), st>>>(
                t.leaf_ids, t.lv, t.start, t.count, c.thr, v0, c.perm, c.x, c.has_masses ? c.m.p : nullptr, c.mass, c.box, c.eps, c.mmax, c.xs64,
                c.xs32);
        }
        VG_LAUNCH_CHECK();
    };
    bool operators = false;  // enqueued
    auto read_back = [&] {
        c.lists_ahead = ahead && cap > 0 && cap <= AHEAD_CELLS;
        if (c.lists_ahead) {
            lists_enqueue(c, SH, cap);
            VG_HIP(hipEventRecord(c.ev_lists, st));
        } else {
            VG_HIP(hipEventRecord(c.ev_tree, st));
        }
        if (ahead && !operators) operators_build(c);
        operators = true;
        wait_host_word(&host->seq, c.tree_seq, st);
        if (host->box[6] != 0) throw Error(2, "non-finite particle coordinates");
    };
    for (;;) {
        ++c.tree_seq;
        sort_and_count();
        if (cap > 0) cells();
        read_back();
        if (hlv[LV_DEEP]) {
            if (SH == MAXD)
                throw Error(3, "octree deeper than 21 levels: more than floor(sqrt(8) s) points closer than the root box / 2^21");
            SH = MAXD;
            continue;
        }
        if (1 + 8ll * hlv[LV_I + SH] <= cap) break;
        cap = 1 + 8ll * hlv[LV_I + SH];
        ensure_cells(t, cap);
        ++c.tree_seq;
        cells();
        read_back();
        break;
    }
    for (int a = 0; a < 6; ++a) t.box[a] = host->box[a];
    t.lvl_off.assign({0, 1});
    t.int_off.assign({0, hlv[LV_I + 1]});
    for (int d = 0; t.int_off[d + 1] > t.int_off[d]; ++d) {
        t.lvl_off.push_back(hlv[d + 2]);
        t.int_off.push_back(hlv[LV_I + d + 2]);
    }
    t.depth = static_cast<int>(t.lvl_off.size()) - 2;
    t.ncells = t.lvl_off.back();
    t.nleaves = hlv[LV_NLEAF];
    if (t.nleaves && c.thr > LS_MAXTHR) {
        k_leaf_sort<<<static_cast<unsigned>(t.nleaves), 256, c.thr * sizeof(uint32_t), st>>>(t.leaf_ids, t.start, t.count, v0, c.perm);
        k_gather<<<ceil_div(n, 256), 256, 0, st>>>(c.perm, n, c.x, c.has_masses ? c.m.p : nullptr, c.mass, c.box, c.eps, c.mmax, c.xs64, c.xs32);
        VG_LAUNCH_CHECK();
        VG_HIP(hipEventRecord(c.lists_ahead ? c.ev_lists : c.ev_tree, st));  // what P2P waits for has these particles in order
    }
    t.ref_valid = false;
}

void lists_build(Ctx &c) { lists_enqueue(c, MAXD, c.t.ncells); }

void ref_numbering(Ctx &c) {
    hipStream_t st = c.stream;
    TreeDev &t = c.t;
    const int64_t nc = t.ncells;
    const int64_t nint = t.int_off.back();
    t.ref_id.ensure(std::max<int64_t>(1, nc));
    if (nint == 0) {
        k_ref_ids<<<ceil_div(nc, 256), 256, 0, st>>>(nc, t.parent, t.octant, nullptr, nullptr, t.ref_id);
        VG_LAUNCH_CHECK();
        t.ref_valid = true;
        return;
    }
    const uint32_t keep = c.thr + 1;
    int pow2 = 1;
    while (static_cast<uint32_t>(pow2) < 8 * keep) pow2 <<= 1;
    if (pow2 * sizeof(uint32_t) > 64 * 1024) throw Error(1, "export of the reference numbering supports floor(sqrt(8) s) < 2048");
    DevBuf<int32_t> int_index, rank;
    int_index.ensure(nc);
    rank.ensure(nint);
    c.slist.ensure(static_cast<size_t>(nint) * keep);
    for (int b = 0; b < 2; ++b) {
        c.rkey[b].ensure(nint);
        c.rval[b].ensure(nint);
    }
    k_int_index<<<ceil_div(nint, 256), 256, 0, st>>>(t.int_ids, nint, int_index);
    for (int d = t.depth; d >= 0; --d) {
        const int64_t a = t.int_off[d], b = t.int_off[d + 1];
        if (b > a)
            k_smallest<<<static_cast<unsigned>(b - a), 256, pow2 * sizeof(uint32_t), st>>>(t.int_ids.p + a, static_cast<int>(b - a), t.child, t.start,
                                                                                            t.count, c.perm, int_index, c.slist, keep, c.rkey[0], c.rval[0],
                                                                                            t.level, pow2);
    }
    VG_LAUNCH_CHECK();
    uint64_t *k0 = c.rkey[0].p, *k1 = c.rkey[1].p;
    uint32_t *v0 = c.rval[0].p, *v1 = c.rval[1].p;
    radix_sort_pairs(st, k0, v0, k1, v1, nint, 0, 64, c.rs_hist);
    k_rank_of<<<ceil_div(nint, 256), 256, 0, st>>>(v0, nint, rank);
    k_ref_ids<<<ceil_div(nc, 256), 256, 0, st>>>(nc, t.parent, t.octant, int_index, rank, t.ref_id);
    VG_LAUNCH_CHECK();
    VG_HIP(hipStreamSynchronize(st));
    t.ref_valid = true;
}

}  // namespace vg
