// p2p.hip - near field (P2P) of every non-empty leaf.
//
// The reference sums, for each point i of a leaf, over every cell of the
// leaf's NI list and over all points of that cell's subtree, skipping i
// itself (fmm.hpp:377-385,513-540, solver_ref.hpp:209-210).  The NI list of a
// cell is its parent's NI list followed by its own new entries
// (solver_ref.hpp:126), so a leaf's list is the concatenation of the local
// entries of its ancestors and itself.  Every subtree is one contiguous range
// of the sorted particles, so each entry is a (start, count) range.
//
// Work items: a plan kernel counts each non-empty leaf's sources and cuts them
// into even chunks, so leaves with long inherited lists spread over many
// wavefronts; each (leaf, chunk) is one item, for one wavefront.
//  * FP32 (k_p2p_mc): squared distances on the matrix cores.
//  * FP64 (k_p2p_f64): pairs by differences.
// A leaf with one chunk writes its result; split leaves write partial sums, a row of
// whole 16-target tiles for each chunk, which L2P adds in chunk order
// (deterministic).  With a nonzero softening the i == j force is exactly zero (dx = dy
// = dz = 0), so it needs no branch; without softening a select removes it.  The i == j
// potential m_i / eps is left out by the particle's index, in the few groups of sources
// that hold targets: subtracted afterwards, it leaves the rounding of sums as large as
// itself (FP32, eps = 1e-4, energy of 17 particles: 8e-6 off, now 1.2e-8; of 120 with one
// mass: 1.1e-6, now 4.5e-8).
#include "gravity.hpp"

namespace vg {
namespace {

constexpr int MAXE = 27 * (MAXD + 1);

// Sources per work item of a leaf cut into nch: even, in whole groups of 64.
__host__ __device__ inline uint32_t chunk_len(uint32_t total, uint32_t nch) { return ((total + nch - 1) / nch + 63) / 64 * 64; }

// ---- FP32: squared distances on the matrix cores -------------------------
//
// What bounds it: VALU issue.  Measured per wavefront instruction on gfx950
// with 4 or more wavefronts per SIMD: FP32 add / mul / fma 2.4-2.9 cycles,
// v_rsq_f32 8.4, other VALU 4.3, v_mfma_f32_4x4x1 8.8; FP32 matrix
// instructions run in the VALU's own FMA units (their times add up), bf16 ones
// beside it.  Differences, squared distance, rsq, cube and three sums cost 11
// FP32 instructions and one rsq for 64 pairs, and the kernel that did so ran
// at that bound: 5.97 ms for the 1.66e10 pairs of the 4M Plummer input.  Here
//   r^2 = |x_j|^2 - 2 x_i x_j + (|x_i|^2 + eps^2)
// is one v_mfma_f32_16x16x32_bf16 per 16 sources x 16 targets: every operand
// is split into three bf16 values that add up to it exactly, and 8 of the 9
// products of the parts (the last is below 2^-32) of the three coordinates and
// the two norms fill 30 of the 32 products of a row.  Then rsq, two products,
// and sum w (x_j - x_i) = sum w x_j - x_i sum w by v_mfma_f32_4x4x1, whose rows
// are (x, y, z, 1) times the source's mass and whose columns are the lanes'
// own w: 2 products and one rsq for 64 pairs beside the 8.8 cycles.  4.26 ms on
// that input; one wavefront per item, without block barriers, and all leaf
// sizes in one launch: 0.85 -> 0.34 ms on a 100k Plummer sphere, 0.30 -> 0.10 ms
// on 8,000 particles.
//
// Range: m x and r^-3 appear by themselves, so lengths and masses far from 1 (SI and
// cgs units) come in units of their own (length_shift, mass_shift).
//
// Error: positions are taken relative to the centre of the targets' box (radius
// R), so at distance d from the box the expansion takes up to 1.5 (R + d)^2 / d^2
// roundings (2^-24) of a pair's force, where differences of positions stored up to D
// from the root centre lose 4 D / d and more to the rounding of these.  Tiles of 16
// sources that come nearer than where the first is the second, (R + d)^2 = 3 D d, within
// R / 8 to R / 2, are left to a second pass by differences, which also has the pairs of a
// particle with itself: R / 8 for leaves small beside D (15 % of the tiles on the 4M
// Plummer input), more for the large ones of shallow trees and of the root's middle.  With
// R / 8 there too a pair was off by up to 107 roundings on positions that FP32 holds
// exactly, now by 13 (differences: 7).  RMS, median and 99.99th percentile of the relative
// force error against the FP64 mode at order 12, differences alone -> R / 8 everywhere -> this:
//   2000 uniform, s = 200      6.3e-7 2.0e-7 1.32e-5   6.1e-7 1.3e-7 1.48e-5   5.7e-7 1.2e-7 1.32e-5
//   8000 Plummer, s = 200      1.41e-6 1.34e-7 4.2e-5  1.42e-6 1.59e-7 4.2e-5  1.40e-6 1.32e-7 4.2e-5
//   2^18 Plummer, s = 64       2.4e-6 3.4e-7 3.7e-5    2.4e-6 2.4e-7 3.7e-5    2.4e-6 2.4e-7 3.7e-5
//   2^18 mixture, s = 64       1.8e-6 4.7e-7 4.7e-5    1.8e-6 3.8e-7 4.7e-5    1.8e-6 3.8e-7 4.7e-5
// (the last two: position rounding).  R / 4 and R / 2 everywhere cost 3 and 7 % of a 4M
// Plummer step, this rule nothing there and 0.7 to 1.4 % of one of 64,000 particles, s = 128.
constexpr float MC_NEAR = 1.0f / 8, MC_NEAR_LARGE = 1.0f / 2;
// 16-target tiles of an item at most: 8 registers a tile and 4 more in flight;
// the potential's mass products take the registers of one (6 there: 0.71
// against 0.66 ms at 2^18 particles)
constexpr int mc_tiles(bool pot) { return pot ? 5 : 6; }
// An item's cost is its target tiles times its 64-source groups: at most 512
// (256 and 1024: +4 % and +0 % on the 4M Plummer input, -10 % and +20 % at 100k
// particles), less with few leaves, and at most 64 groups, one per lane of the
// entry table.
constexpr uint32_t MC_COST = 512, MC_MINCOST = 16;
// FP64 items: 4 tiles at most (28 registers a tile, 6 spilled), and smaller ones with
// fewer leaves than 64 per CU (16, 32 and 64: 198, 134 and 111 us at 16384 particles in leaves of
// 18; least costs of 4, 8 and 16 alike).
constexpr int F64_TILES = 4, F64_LEAVES = 64;
constexpr uint32_t F64_MINCOST = 16;
constexpr uint32_t MC_CHUNK = 64 * 64;
// Rows of partial sums of a leaf at most: 12, or as many as keep all particles' rows
// within 3 2^20 entries (48 MB, FP64 96), or one for 16 sources of each particle (leaves of
// few particles with long lists; of up to 4096 particles).  Where an item then has more
// than MC_CHUNK sources (leaves of thousands of particles), as many launches as that takes
// add to its row.  A context's memory in GB with rows as long as the largest leaf for every
// 512 to 4096 sources, and with these: FP64, 2^19 Plummer particles with s = 2000, 34.5 ->
// 0.46; 2^20 uniform, s = 5000, 17.6 -> 0.92, FP32 4.6 -> 0.62; evaluations 59 -> 56, 28.2 -> 27.7
// and 11.3 -> 11.6 ms (the last with the wider near pass above).
constexpr uint32_t PART_ROWS = 12, PART_ENTRIES = 3u << 20, PART_MAXLEAF = 4096;
// A leaf's targets go to items of at most mt tiles, evenly.
__host__ __device__ inline uint32_t mc_batches(uint32_t nt, int mt) { return ((nt + 15) / 16 + mt - 1) / mt; }
__host__ __device__ inline uint32_t mc_batch_tiles(uint32_t nt, int mt) { return ((nt + 15) / 16 + mc_batches(nt, mt) - 1) / mc_batches(nt, mt); }
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// [upper 16 bits of lo, upper 16 bits of hi]: two bf16 values cut off (not rounded)
__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) { return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u); }
__device__ __forceinline__ float cut_bf16(float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); }
// x = h + m + l with three bf16 values, exactly (3 x 8 of the 24 bits): h, m
// and l are the upper halves of x, r1 and r2.
struct Split3 {
    float x, r1, r2;
    __device__ __forceinline__ explicit Split3(float v) : x(v), r1(v - cut_bf16(v)), r2(r1 - cut_bf16(r1)) {}
    __device__ __forceinline__ uint32_t hm() const { return pk_bf16(x, r1); }
    __device__ __forceinline__ uint32_t hh() const { return pk_bf16(x, x); }
    __device__ __forceinline__ uint32_t mm() const { return pk_bf16(r1, r1); }
    __device__ __forceinline__ uint32_t ll() const { return pk_bf16(r2, r2); }
};
constexpr uint32_t BF16_ONES = 0x3f803f80u;

struct McLds {
    uint4 P[4][64];        // 64 staged sources: bf16 operand, one 16-byte group per 16 lanes of the product
    float4 Q[64];          // m (x, y, z, 1) of the staged sources; (x, y, z, m) in the near pass; while the entries are laid out, their masks
    int32_t delta[MAXE];   // per entry of the item: particle index minus position in the item
    uint16_t near[64 * 4]; // 16-source tiles left to the near pass
    float4 M[16];          // for the potential: masses of the staged sources; in the near pass, their indices
};

// A work item as the plan leaves it.
struct alignas(32) McWork {
    int32_t cell, level;  // the leaf
    uint32_t pt0, nt;     // its targets: particles pt0 .. pt0 + nt - 1, of the leaf's from t0 on
    uint32_t src0, len;   // its share of the leaf's sources
    uint32_t out;         // first tile of this share's row of partial sums, ~0: the only share
    uint32_t t0;
};

// The piece of the item that a launch takes: MC_CHUNK of its sources; false if there is none.
__device__ __forceinline__ bool take_piece(McWork &wk, uint32_t piece) {
    const uint32_t at = piece * MC_CHUNK;
    if (piece && at >= wk.len) return false;
    wk.src0 += at;
    wk.len = min(MC_CHUNK, wk.len - at);
    return true;
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Where a work item's sources lie: lane g has, of the item's group of 64 sources g,
// the entry of the first one and where entries begin in it.
struct Sources {
    uint32_t mlo, mhi;  // the begins, from the group's second source on
    int rank;           // entry of the group's first source
};
__device__ __forceinline__ Sources lay_out_entries(const McWork &wk, int32_t *delta, uint64_t *mask, const uint32_t *__restrict__ start,
                                                   const uint32_t *__restrict__ count, const int32_t *__restrict__ anc, const int32_t *__restrict__ ni,
                                                   const int32_t *__restrict__ ni_cnt) {
    const int lane = threadIdx.x, lev = wk.level;
    const int32_t c = wk.cell;
    Sources I;
    mask[lane] = 0;
    // the leaf's NI list: its ancestors' own entries, root first; lane l has ancestor l
    const int32_t an = lane <= lev ? anc[static_cast<int64_t>(c) * (MAXD + 1) + lane] : 0;
    const int an_cnt = lane <= lev ? ni_cnt[an] : 0;
    int an_end = an_cnt;
    for (int d = 1; d < 32; d <<= 1) {
        const int o = __shfl_up(an_end, d, 64);
        if (lane >= d) an_end += o;
    }
    const int E = __builtin_amdgcn_readlane(an_end, lev);
    const uint64_t live = __ballot(an_cnt > 0);
    auto entry = [&](int e, uint32_t &st, uint32_t &cn) {  // particle range of entry e
        int l = 0;
        for (uint64_t w = live; w; w &= w - 1) {  // the last ancestor with entries whose first one is <= e
            const int k = __builtin_ctzll(w);
            if (__builtin_amdgcn_readlane(an_end - an_cnt, k) <= e) l = k;
        }
        const int32_t a = __shfl(an, l, 64);
        const int o = e - __shfl(an_end - an_cnt, l, 64);
        st = cn = 0;
        if (e < E) {
            const int32_t cell = ni[27 * static_cast<int64_t>(a) + o];
            st = start[cell];
            cn = count[cell];
        }
    };
    // the entries that reach into [src0, src1), empty ones dropped, and where they begin in it
    const uint32_t src0 = wk.src0, src1 = src0 + wk.len;
    wave_lds_sync();
    uint32_t carry = 0, st, cn;
    int kept = 0;
    entry(lane, st, cn);
    for (int e0 = 0; e0 < E && carry < src1; e0 += 64) {
        uint32_t nst = 0, ncn = 0;
        if (e0 + 64 < E) entry(e0 + 64 + lane, nst, ncn);  // on its way while this run is laid out
        uint32_t incl = cn;
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        const uint32_t off = carry + incl - cn;
        const bool in = cn > 0 && off + cn > src0 && off < src1;
        const uint64_t bal = __ballot(in);
        if (in) {
            delta[kept + __popcll(bal & ((1ull << lane) - 1))] = static_cast<int32_t>(st - (off - src0));
            const uint32_t o = max(off, src0) - src0;
            atomicOr(reinterpret_cast<unsigned long long *>(&mask[o >> 6]), 1ull << (o & 63));
        }
        kept += __popcll(bal);
        carry += __builtin_amdgcn_readlane(incl, 63);
        st = nst, cn = ncn;
    }
    wave_lds_sync();
    {  // lane g: the entry of group g's first source, and the later begins shifted so that mbcnt counts them
        const uint64_t m = mask[lane];
        const int own = __popcll(m);
        int incl = own;
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        I.rank = incl - own + static_cast<int>(m & 1) - 1;
        I.mlo = static_cast<uint32_t>(m >> 1);
        I.mhi = static_cast<uint32_t>(m >> 33);
    }
    wave_lds_sync();
    return I;
}
// Particle of source `lane` of group g (the last one again past len).
__device__ __forceinline__ int32_t source_of(const Sources &S, const int32_t *delta, int g, uint32_t len) {
    const uint32_t lo = __builtin_amdgcn_readlane(S.mlo, g), hi = __builtin_amdgcn_readlane(S.mhi, g);
    const int e = __builtin_amdgcn_readlane(S.rank, g) + __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
    return delta[e] + static_cast<int32_t>(min(64u * g + threadIdx.x, len - 1));
}

// What a wavefront knows of its work item.
struct McItem {
    const float4 *xs;     // sorted particles (x, y, z relative to the root centre, m)
    uint32_t len;         // sources
    Sources src;
    uint32_t pt0;         // first target
    int nt;               // targets
    float cell;           // half diagonal of the leaf
    float eps2;
    bool um;              // one mass: m1 here, the sums are scaled once
    float m1;             // a power of two, 1 in ordinary units
    bool big;             // squared distances may leave the FP32 range
};

// The item's T tiles of 16 targets against its sources; emit(t, v) gets target
// t's sums (force xyz, potential), in one lane.
template <int T, bool POT, class F>
__device__ __forceinline__ void mc_pass(const McItem &I, McLds &S, F &&emit) {
    const int lane = threadIdx.x, col = lane & 15, quad = lane >> 4;
    const int ng = static_cast<int>((I.len + 63) / 64);
    const float4 first = I.xs[I.pt0];
    float cx = first.x, cy = first.y, cz = first.z;
    auto target = [&](int t) {  // columns past the last target repeat it and are dropped
        const float4 v = I.xs[I.pt0 + min(16 * t + col, I.nt - 1)];
        return float3{v.x - cx, v.y - cy, v.z - cz};
    };
    // box of the targets, relative to the first one; its centre is the origin from here on
    float hx, hy, hz, ns;
    {
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const float3 x = target(t);
            lo[0] = fminf(lo[0], x.x), hi[0] = fmaxf(hi[0], x.x);
            lo[1] = fminf(lo[1], x.y), hi[1] = fmaxf(hi[1], x.y);
            lo[2] = fminf(lo[2], x.z), hi[2] = fmaxf(hi[2], x.z);
        }
#pragma unroll
        for (int a = 0; a < 3; ++a)
            for (int d = 1; d < 16; d <<= 1) {
                lo[a] = fminf(lo[a], __shfl_xor(lo[a], d, 64));
                hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], d, 64));
            }
        cx += 0.5f * (lo[0] + hi[0]), cy += 0.5f * (lo[1] + hi[1]), cz += 0.5f * (lo[2] + hi[2]);
        hx = 0.5f * (hi[0] - lo[0]), hy = 0.5f * (hi[1] - lo[1]), hz = 0.5f * (hi[2] - lo[2]);
        // sources up to near from the box are near; ns = 1 / (2 near), 0 where all are
        const float r = sqrtf(hx * hx + hy * hy + hz * hz);
        // (r + d)^2 = 3 D d at d = e - sqrt(e^2 - r^2), e = 3/2 D - r: r / 2 at e = 5/4 r
        const float e = 1.5f * fmaxf(fmaxf(fabsf(cx) + hx, fabsf(cy) + hy), fabsf(cz) + hz) - r;
        const float even = e > 1.25f * r ? fmaxf(MC_NEAR * r, e - sqrtf(e * e - r * r)) : MC_NEAR_LARGE * r;
        const float nearest = fmaxf(fmaxf(even, I.cell * 0.0078125f), 0x1p-40f);  // r^-3 up to 2^120
        ns = r < 1e18f ? 0.5f / nearest : 0.0f;
        hx = -ns * (hx + I.cell * 1e-5f), hy = -ns * (hy + I.cell * 1e-5f), hz = -ns * (hz + I.cell * 1e-5f);
    }
    asm volatile("" ::: "memory");  // the targets are read again, not kept in registers
    bf8 b[T];
    f4 acc[T];
    float pot[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const float3 x = target(t);
        const Split3 v(quad == 0 ? -2.0f * x.x : quad == 1 ? -2.0f * x.y : quad == 2 ? -2.0f * x.z : x.x * x.x + x.y * x.y + x.z * x.z + I.eps2);
        const uint4 w = quad < 3 ? uint4{v.hh(), v.mm(), v.ll(), v.hm()} : uint4{BF16_ONES, pk_bf16(1.0f, v.x), pk_bf16(v.r1, v.r2), 0u};
        b[t] = __builtin_bit_cast(bf8, w);
        acc[t] = f4{0, 0, 0, 0};
        pot[t] = 0;
    }
    const float *Qw = reinterpret_cast<const float *>(S.Q);
    const f4 zero = {0, 0, 0, 0};
    // far pass: groups of 64 sources, near tiles put aside
    auto source = [&](int g) { return I.xs[source_of(I.src, S.delta, g, I.len)]; };  // this lane's source of group g
    uint32_t mynear = 0;  // lane g: near tiles of group g
    float4 nx = source(0);
    for (int g = 0; g < ng; ++g) {
        float x = nx.x - cx, y = nx.y - cy, z = nx.z - cz;
        float m = I.um ? I.m1 : nx.w;
        if (g + 1 < ng)
            nx = source(g + 1);
        else if (64u * g + lane >= I.len)  // the last source again, without mass
            m = 0.0f;
        auto out01 = [&](float v, float h) { return __builtin_amdgcn_fmed3f(fmaf(fabsf(v), ns, h), 0.0f, 1.0f); };
        const float ex = out01(x, hx), ey = out01(y, hy), ez = out01(z, hz);
        const uint64_t near = __ballot(ex * ex + ey * ey + ez * ez <= 0.25f);
        uint32_t nib = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) nib |= ((near >> (16 * k)) & 0xffff) ? 1u << k : 0u;
        if (nib) {
            mynear = lane == g ? nib : mynear;
            if (nib == 15) continue;
        }
        float n2 = x * x + y * y + z * z;
        if (I.big && !(n2 < 1e37f)) x = y = z = m = 0.0f, n2 = 1e37f;  // a source that far away pulls with 0 in FP32
        __builtin_amdgcn_wave_barrier();  // the last group's reads come before these writes (one wavefront's LDS accesses keep their order)
        const Split3 sx(x), sy(y), sz(z), sn(n2);
        S.P[0][lane] = uint4{sx.hm(), sx.hm(), sx.hm(), sx.ll()};
        S.P[1][lane] = uint4{sy.hm(), sy.hm(), sy.hm(), sy.ll()};
        S.P[2][lane] = uint4{sz.hm(), sz.hm(), sz.hm(), sz.ll()};
        S.P[3][lane] = uint4{sn.hm(), pk_bf16(sn.r2, 1.0f), BF16_ONES, 0u};
        S.Q[lane] = float4{m * x, m * y, m * z, m};
        if (POT) reinterpret_cast<float *>(S.M)[lane] = m;
        wave_lds_sync();
        auto distances = [&](int k, f4 *r) {
            const bf8 a = __builtin_bit_cast(bf8, S.P[quad][16 * k + col]);
#pragma unroll
            for (int t = 0; t < T; ++t) r[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[t], zero, 0, 0, 0);
        };
        auto sums = [&](int k, float q, f4 *r) {
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) r[t][i] = rsq(r[t][i]);
            if (POT) {
                const float4 m4 = S.M[4 * k + quad];
#pragma unroll
                for (int t = 0; t < T; ++t) pot[t] += m4.x * r[t][0] + m4.y * r[t][1] + m4.z * r[t][2] + m4.w * r[t][3];
            }
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) r[t][i] = r[t][i] * r[t][i] * r[t][i];
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(q, r[t][0], acc[t], 2, 0, 0);
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(q, r[t][1], acc[t], 2, 1, 0);
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(q, r[t][2], acc[t], 2, 2, 0);
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(q, r[t][3], acc[t], 2, 3, 0);
        };
#pragma unroll 1
        for (int k = 0; k < 4; ++k) {
            if (nib >> k & 1) continue;
            f4 r[T];
            const float q = Qw[64 * k + lane];
            distances(k, r);
            sums(k, q, r);
            // all rsq, then the products, then the sums: 4.69 -> 4.52 ms on the 4M Plummer input against the compiler's order
            __builtin_amdgcn_sched_group_barrier(0x400, 4 * T, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, (POT ? 12 : 8) * T, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 4 * T, 0);
        }
    }
    asm volatile("" ::: "memory");
    // sum m w (x_j - x_i) = sum m w x_j - x_i sum m w; from here on positions are as stored
    float xt[T], yt[T], zt[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const float3 x = target(t);
        acc[t][0] -= x.x * acc[t][3];
        acc[t][1] -= x.y * acc[t][3];
        acc[t][2] -= x.z * acc[t][3];
        acc[t][3] = pot[t];
    }
    cx = cy = cz = 0.0f;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const float3 x = target(t);
        xt[t] = x.x, yt[t] = x.y, zt[t] = x.z;
    }
    // near pass: four 16-source tiles at a time, by differences
    int nn;
    {
        int incl = __builtin_popcount(mynear);
        const int own = incl;
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        nn = __builtin_amdgcn_readlane(incl, 63);
        int at = incl - own;
        for (int k = 0; k < 4; ++k)
            if (mynear >> k & 1) S.near[at++] = static_cast<uint16_t>(4 * lane + k);
        wave_lds_sync();
    }
    int ni = 0;  // particle index of nx
    auto near_source = [&](int j) {  // this lane's source of the near tiles 4 j .. 4 j + 3
        const int n = 4 * j + quad;
        const int tl = S.near[min(n, nn - 1)], g = tl >> 2, pos = 16 * (tl & 3) + col;
        const uint64_t m = static_cast<uint64_t>(static_cast<uint32_t>(__shfl(static_cast<int>(I.src.mhi), g, 64))) << 32 | static_cast<uint32_t>(__shfl(static_cast<int>(I.src.mlo), g, 64));
        const int e = __shfl(I.src.rank, g, 64) + __popcll(m & ((1ull << pos) - 1));
        const uint32_t f = 64u * g + pos;
        ni = S.delta[e] + static_cast<int32_t>(min(f, I.len - 1));
        float4 v = I.xs[ni];
        if (I.um) v.w = I.m1;
        if (n >= nn || f >= I.len) v.w = 0.0f;
        return v;
    };
    if (nn > 0) nx = near_source(0);
    for (int j = 0; 4 * j < nn; ++j) {
        __builtin_amdgcn_wave_barrier();
        S.Q[lane] = nx;
        const int who = ni - static_cast<int>(I.pt0);  // the target that it is
        if (POT) reinterpret_cast<int *>(S.M)[lane] = who;
        const bool own = POT && __ballot(who >= 0 && who < I.nt) != 0;  // the few tiles that hold targets
        if (4 * j + 4 < nn) nx = near_source(j + 1);
        wave_lds_sync();
        const int kn = min(4, nn - 4 * j);
        auto pairs = [&](auto soft, auto own) {
#pragma unroll 1
            for (int k = 0; k < kn; ++k) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4 s = S.Q[16 * k + 4 * quad + i];
                    const int self = decltype(own)::value ? reinterpret_cast<const int *>(S.M)[16 * k + 4 * quad + i] - col : 0;
#pragma unroll
                    for (int t = 0; t < T; ++t) {
                        const float dx = s.x - xt[t], dy = s.y - yt[t], dz = s.z - zt[t];
                        const float r2 = I.eps2 + dx * dx + dy * dy + dz * dz;
                        float ri = rsq(r2);
                        if (!decltype(soft)::value) ri = r2 > 0.0f ? ri : 0.0f;  // a particle and itself
                        const float mr = s.w * ri, w = mr * ri * ri;
                        acc[t][0] += w * dx;
                        acc[t][1] += w * dy;
                        acc[t][2] += w * dz;
                        if (POT) acc[t][3] += decltype(own)::value && self == 16 * t ? 0.0f : mr;
                    }
                }
            }
        };
        if (!(I.eps2 > 0.0f))
            pairs(std::false_type{}, std::false_type{});
        else if (POT && own)
            pairs(std::true_type{}, std::bool_constant<POT>{});
        else
            pairs(std::true_type{}, std::false_type{});
    }
    // the four lane groups hold the sums over their own source rows
#pragma unroll
    for (int t = 0; t < T; ++t) {
#pragma unroll
        for (int j = 0; j < (POT ? 4 : 3); ++j) {
            acc[t][j] += __shfl_xor(acc[t][j], 16, 64);
            acc[t][j] += __shfl_xor(acc[t][j], 32, 64);
        }
        if (quad == 0 && 16 * t + col < I.nt) emit(16 * t + col, acc[t]);
    }
}

// One wavefront per work item.
template <bool POT>
__global__ __launch_bounds__(64, 4) void k_p2p_mc(const McWork *__restrict__ items, const uint32_t *__restrict__ start,
                                                       const uint32_t *__restrict__ count, const int32_t *__restrict__ anc,
                                                       const int32_t *__restrict__ ni, const int32_t *__restrict__ ni_cnt,
                                                       const double *__restrict__ bmin, const double *__restrict__ bmax, const float4 *__restrict__ xs,
                                                       float eps2, float G, bool um, float m1, bool big, float fscale, float pscale,
                                                       float4 *__restrict__ acc, float4 *__restrict__ partial, float unit, uint32_t piece) {
    __shared__ McLds S;
    McWork wk = items[blockIdx.x];
    if (!take_piece(wk, piece)) return;
    const int32_t c = wk.cell;
    const int lane = threadIdx.x;
    McItem I;
    I.nt = static_cast<int>(wk.nt);
    I.pt0 = wk.pt0;
    I.len = wk.len;
    I.src = lay_out_entries(wk, S.delta, reinterpret_cast<uint64_t *>(S.Q), start, count, anc, ni, ni_cnt);
    I.xs = xs;
    const double lx = bmin[3ll * c], ly = bmin[3ll * c + 1], lz = bmin[3ll * c + 2], ux = bmax[3ll * c], uy = bmax[3ll * c + 1], uz = bmax[3ll * c + 2];
    const float wx = static_cast<float>(ux - lx) * unit, wy = static_cast<float>(uy - ly) * unit, wz = static_cast<float>(uz - lz) * unit;
    I.cell = 0.5f * sqrtf(wx * wx + wy * wy + wz * wz);
    I.eps2 = eps2;
    I.um = um;
    I.m1 = m1;
    I.big = big;
    float4 *out = wk.out != ~0u ? partial + static_cast<size_t>(wk.out) * 16 : nullptr;
    auto emit = [&](int t, const f4 &v) {
        const float sx = v[0] * fscale, sy = v[1] * fscale, sz = v[2] * fscale, sp = v[3] * pscale;
        if (out) {
            float4 o = float4{sx, sy, sz, sp};
            if (piece) {
                const float4 u = out[wk.t0 + t];
                o.x += u.x, o.y += u.y, o.z += u.z, o.w += u.w;
            }
            out[wk.t0 + t] = o;
        } else {
            acc[I.pt0 + t] = float4{G * sx, G * sy, G * sz, sp};
        }
    };
    if (wk.len == 0) {  // a last chunk that the even lengths left empty
        for (int t = lane; t < I.nt; t += 64) emit(t, f4{0, 0, 0, 0});
        return;
    }
    constexpr int MT = mc_tiles(POT);
    const int T = (I.nt + 15) / 16;  // at most MT
    if (T == 1)
        mc_pass<1, POT>(I, S, emit);
    else if (T == 2)
        mc_pass<2, POT>(I, S, emit);
    else if (T == 3)
        mc_pass<3, POT>(I, S, emit);
    else if (T == 4)
        mc_pass<4, POT>(I, S, emit);
    else if (T == 5)
        mc_pass<5, POT>(I, S, emit);
    else
        mc_pass<MT, POT>(I, S, emit);
}

// ---- FP64 ----------------------------------------------------------------
//
// One wavefront per work item as above; pairs by differences, 64 sources at a time
// through LDS, the 16 lanes of a group holding T targets each and the four groups
// taking every fourth source.  Bound by FP64 issue (4.6 cycles): 16 operations and
// one v_rsq_f64 (16 cycles) for 64 pairs.  Per evaluation, against a 256-thread
// block per 1024 to 16384 sources, a launch per leaf size one after the other, and
// two Newton steps for each root: 16384 particles (s = 64) 0.33 -> 0.15 ms, 64k
// mixture 1.05 -> 0.40, 128k (s = 128) 3.0 -> 1.7, 1M 3.3 -> 2.7 ms.
template <int T, bool POT, class F>
__device__ __forceinline__ void f64_pass(const double4 *__restrict__ xs, const Sources &src, const int32_t *delta, double4 *tile, int *who, uint32_t len,
                                         uint32_t pt0, int nt, double eps2, bool um, F &&emit) {
    const int lane = threadIdx.x, col = lane & 15, quad = lane >> 4;
    const int ng = static_cast<int>((len + 63) / 64);
    double x[T], y[T], z[T], acc[T][4];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const double4 v = xs[pt0 + min(16 * t + col, nt - 1)];  // columns past the last target repeat it and are dropped
        x[t] = v.x, y[t] = v.y, z[t] = v.z;
        acc[t][0] = acc[t][1] = acc[t][2] = acc[t][3] = 0;
    }
    int ni = source_of(src, delta, 0, len);  // particle index of nx
    double4 nx = xs[ni];
    for (int g = 0; g < ng; ++g) {
        __builtin_amdgcn_wave_barrier();
        const bool full = 64u * g + 64 <= len;
        if (um) nx.w = 1.0;
        if (64u * g + lane >= len) nx.w = 0.0;  // the last source again, without mass
        tile[lane] = nx;
        const int me = ni - static_cast<int>(pt0);  // the target that it is
        if (POT) who[lane] = me;
        const bool own = POT && __ballot(me >= 0 && me < nt) != 0;  // the few groups that hold targets
        if (g + 1 < ng) {
            ni = source_of(src, delta, g + 1, len);
            nx = xs[ni];
        }
        wave_lds_sync();
        auto pairs = [&](auto soft, auto weighted, auto own) {
#pragma unroll 2
            for (int i = 0; i < 16; ++i) {
                const double4 s = tile[4 * i + quad];
                const int self = decltype(own)::value ? who[4 * i + quad] - col : 0;
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const double dx = s.x - x[t], dy = s.y - y[t], dz = s.z - z[t];
                    const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, eps2)));
                    const double h = __builtin_amdgcn_rsq(r2);  // 2^-24 at worst; r2^(-3/2) = h^3 (1 + 3/2 e + 15/8 e^2 + ..), e^3 below 2^-69
                    const double hh = h * h, e = fma(-r2, hh, 1.0);
                    const double c = (decltype(weighted)::value ? h * s.w : h) * hh;
                    double w = fma(c * e, fma(e, 1.875, 1.5), c);
                    if (!decltype(soft)::value) w = r2 > 0.0 ? w : 0.0;  // a particle and itself
                    acc[t][0] = fma(w, dx, acc[t][0]);
                    acc[t][1] = fma(w, dy, acc[t][1]);
                    acc[t][2] = fma(w, dz, acc[t][2]);
                    if (POT) {
                        double ri = fma(h * e, fma(e, 0.375, 0.5), h);
                        if (!decltype(soft)::value) ri = r2 > 0.0 ? ri : 0.0;
                        if (decltype(own)::value) ri = self == 16 * t ? 0.0 : ri;
                        acc[t][3] = decltype(weighted)::value ? fma(s.w, ri, acc[t][3]) : acc[t][3] + ri;
                    }
                }
            }
        };
        if (eps2 > 0.0) {
            if (POT && own)
                pairs(std::true_type{}, std::true_type{}, std::bool_constant<POT>{});
            else if (um && full)
                pairs(std::true_type{}, std::false_type{}, std::false_type{});
            else
                pairs(std::true_type{}, std::true_type{}, std::false_type{});
        } else {
            if (um && full)
                pairs(std::false_type{}, std::false_type{}, std::false_type{});
            else
                pairs(std::false_type{}, std::true_type{}, std::false_type{});
        }
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
#pragma unroll
        for (int j = 0; j < (POT ? 4 : 3); ++j) {
            acc[t][j] += __shfl_xor(acc[t][j], 16, 64);
            acc[t][j] += __shfl_xor(acc[t][j], 32, 64);
        }
        if (quad == 0 && 16 * t + col < nt) emit(16 * t + col, acc[t]);
    }
}

template <bool POT>
__global__ __launch_bounds__(64, 4) void k_p2p_f64(const McWork *__restrict__ items, const uint32_t *__restrict__ start,
                                                   const uint32_t *__restrict__ count, const int32_t *__restrict__ anc, const int32_t *__restrict__ ni,
                                                   const int32_t *__restrict__ ni_cnt, const double4 *__restrict__ xs, double eps2, double G, bool um,
                                                   double mu, double4 *__restrict__ acc, double4 *__restrict__ partial, uint32_t piece) {
    __shared__ double4 tile[64];
    __shared__ int32_t delta[MAXE], who[POT ? 64 : 1];
    McWork wk = items[blockIdx.x];
    if (!take_piece(wk, piece)) return;
    const int lane = threadIdx.x, nt = static_cast<int>(wk.nt);
    const double sc = um ? mu : 1.0;
    double4 *out = wk.out != ~0u ? partial + static_cast<size_t>(wk.out) * 16 : nullptr;
    const Sources src = lay_out_entries(wk, delta, reinterpret_cast<uint64_t *>(tile), start, count, anc, ni, ni_cnt);
    auto emit = [&](int t, const double *v) {
        const double sx = v[0] * sc, sy = v[1] * sc, sz = v[2] * sc, sp = v[3] * sc;
        if (out) {
            double4 o = double4{sx, sy, sz, sp};
            if (piece) {
                const double4 u = out[wk.t0 + t];
                o.x += u.x, o.y += u.y, o.z += u.z, o.w += u.w;
            }
            out[wk.t0 + t] = o;
        } else {
            acc[wk.pt0 + t] = double4{G * sx, G * sy, G * sz, sp};
        }
    };
    if (wk.len == 0) {  // a last chunk that the even lengths left empty
        const double none[4] = {0, 0, 0, 0};
        for (int t = lane; t < nt; t += 64) emit(t, none);
        return;
    }
    const int T = (nt + 15) / 16;  // at most F64_TILES
    auto pass = [&](auto tiles) { f64_pass<decltype(tiles)::value, POT>(xs, src, delta, tile, who, wk.len, wk.pt0, nt, eps2, um, emit); };
    if (T == 1)
        pass(std::integral_constant<int, 1>{});
    else if (T == 2)
        pass(std::integral_constant<int, 2>{});
    else if (T == 3)
        pass(std::integral_constant<int, 3>{});
    else
        pass(std::integral_constant<int, F64_TILES>{});
}

// Leaf classes, by the cost of their items (16-target tiles times 64-source
// groups): class j costs at least 2^(8 - j), so the largest start first.
constexpr int NCLS = 7;
constexpr int NSC = NCLS + 2;  // scanned per leaf: tiles of partial sums, items of each class, split flag
constexpr int NBT = NSC + 1;   // words of a plan block: their totals, and the most pieces of an item
__device__ inline int leaf_class(uint32_t nt, uint32_t src, uint32_t nch, int mt) {
    const uint32_t cost = mc_batch_tiles(nt, mt) * (chunk_len(src, nch) / 64);
    return max(0, min(NCLS - 1, 8 - (31 - __builtin_clz(max(cost, 1u)))));
}

// Per leaf: source count -> chunks (of at most chunk target tiles times source
// groups) and class; block-local exclusive scans of
// the NSC components (one leaf per thread, 256 per block) and block totals.
__global__ __launch_bounds__(256) void k_p2p_plan(const int32_t *__restrict__ leaves, int nleaves, const int8_t *__restrict__ level,
                                                  const uint32_t *__restrict__ count, const int32_t *__restrict__ anc, const uint32_t *__restrict__ local,
                                                  uint32_t *__restrict__ nchunk, uint32_t *__restrict__ cls, uint32_t *__restrict__ nsrc, uint32_t *__restrict__ pre,
                                                  uint32_t *__restrict__ btot, uint32_t chunk, int mt, uint32_t minrow,
                                                  uint32_t maxrows) {
    __shared__ uint32_t wtot[4][NSC], s_pieces;
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (threadIdx.x == 0) s_pieces = 1;
    __syncthreads();
    const unsigned lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t v[NSC] = {};
    if (k < nleaves) {
        const int32_t c = leaves[k];
        uint32_t src = 0;
        for (int l = 0; l <= level[c]; ++l) src += local[anc[static_cast<int64_t>(c) * (MAXD + 1) + l]];
        const uint32_t nt = count[c];
        // as many groups as the cost allows, but no fewer than minrow eighths of the tiles (the rows of partial sums of a large leaf stay few)
        const uint32_t lim = 64 * min(MC_CHUNK / 64, max(1 + (nt + 15) / 16 * minrow / 8, chunk / mc_batch_tiles(nt, mt)));
        const uint32_t nch = min(max(maxrows, src / (16 * min(nt, PART_MAXLEAF)) + 1), max(1u, (src + lim - 1) / lim));
        nchunk[k] = nch;
        nsrc[k] = src;
        const uint32_t nit = nch * mc_batches(nt, mt);
        v[0] = nch > 1 ? nch * ((nt + 15) / 16) : 0u;
        const int cl = leaf_class(nt, src, nch, mt);
        cls[k] = cl;
#pragma unroll
        for (int q = 0; q < NCLS; ++q) v[1 + q] = q == cl ? nit : 0u;
        v[NSC - 1] = nch > 1 ? 1u : 0u;
        if (chunk_len(src, nch) > MC_CHUNK) atomicMax(&s_pieces, (chunk_len(src, nch) + MC_CHUNK - 1) / MC_CHUNK);
    }
    uint32_t inc[NSC];
#pragma unroll
    for (int q = 0; q < NSC; ++q) {
        uint32_t x = v[q];
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(x, d, 64);
            if (lane >= static_cast<unsigned>(d)) x += o;
        }
        inc[q] = x;
        if (lane == 63) wtot[w][q] = x;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NSC; ++q) {
        uint32_t base = 0;
        for (unsigned u = 0; u < w; ++u) base += wtot[u][q];
        if (k < nleaves) pre[static_cast<int64_t>(k) * NSC + q] = base + inc[q] - v[q];
        if (threadIdx.x == 255) btot[blockIdx.x * NBT + q] = base + inc[q];
    }
    if (threadIdx.x == 255) btot[blockIdx.x * NBT + NSC] = s_pieces;
}

// One block: exclusive scan of the block totals; writes the class counts and
// bases, the item total and the split-leaf total into scal:
//   scal[0..NCLS) items per class, scal[NCLS..2 NCLS) class bases,
//   scal[2 NCLS] tiles of partial sums, scal[2 NCLS + 1] split leaves, scal[2 NCLS + 2] the
//   most pieces of an item.
// host: the same in pinned host memory, then seq in its last word.
__global__ __launch_bounds__(256) void k_p2p_plan_blocks(uint32_t *__restrict__ btot, int nblocks, uint32_t *__restrict__ scal, uint32_t *host, uint32_t seq) {
    // exclusive scan of each component over the plan blocks, one wavefront per
    // component (wavefront-wide inclusive scans, carried across runs of 64)
    __shared__ uint32_t tot[NSC], s_pieces;
    const unsigned lane = threadIdx.x & 63;
    for (int q = threadIdx.x >> 6; q < NSC; q += 4) {
        uint32_t carry = 0;
        for (int b0 = 0; b0 < nblocks; b0 += 64) {
            const int b = b0 + static_cast<int>(lane);
            const uint32_t v = b < nblocks ? btot[b * NBT + q] : 0u;
            uint32_t x = v;
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t o = __shfl_up(x, d, 64);
                if (lane >= static_cast<unsigned>(d)) x += o;
            }
            if (b < nblocks) btot[b * NBT + q] = carry + x - v;
            carry += __shfl(x, 63, 64);
        }
        if (lane == 0) tot[q] = carry;
    }
    if (threadIdx.x == 0) s_pieces = 1;
    __syncthreads();
    for (int b = threadIdx.x; b < nblocks; b += 256)
        if (btot[b * NBT + NSC] > 1) atomicMax(&s_pieces, btot[b * NBT + NSC]);
    __syncthreads();
    if (threadIdx.x < 2 * NCLS + 3) {  // scal: [class items] [class bases] tiles, split leaves, pieces
        const int j = threadIdx.x;
        uint32_t v = 0;
        if (j < NCLS)
            v = tot[1 + j];
        else if (j < 2 * NCLS)
            for (int k = 0; k < j - NCLS; ++k) v += tot[1 + k];
        else
            v = j == 2 * NCLS ? tot[0] : j == 2 * NCLS + 1 ? tot[NSC - 1] : s_pieces;
        scal[j] = v;
        host[j] = v;
        __threadfence_system();
        if (j == 0) __hip_atomic_store(host + 2 * NCLS + 3, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);  // behind this wavefront's stores
    }
}

// The work items, bucketed by class in leaf order, each with what its wavefront needs
// to start, and where the leaves' partial sums begin.
__global__ __launch_bounds__(256) void k_p2p_items(const int32_t *__restrict__ leaves, int nleaves, const int8_t *__restrict__ level,
                                                      const uint32_t *__restrict__ start, const uint32_t *__restrict__ count,
                                                      const uint32_t *__restrict__ lcls, const uint32_t *__restrict__ nchunk,
                                                      const uint32_t *__restrict__ nsrc, const uint32_t *__restrict__ pre,
                                                      const uint32_t *__restrict__ boff, const uint32_t *__restrict__ scal,
                                                      uint32_t *__restrict__ item_off, McWork *__restrict__ items, int mt) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= nleaves) return;
    const uint32_t *pk = pre + static_cast<int64_t>(k) * NSC;
    const uint32_t *bk = boff + blockIdx.x * NBT;
    const uint32_t nch = nchunk[k], off = bk[0] + pk[0], src = nsrc[k], per = chunk_len(src, nch);
    item_off[k] = off;
    const int cls = lcls[k];
    const int32_t c = leaves[k];
    const uint32_t nt = count[c], pt0 = start[c], bt = 16 * mc_batch_tiles(nt, mt);
    McWork *it = items + scal[NCLS + cls] + bk[1 + cls] + pk[1 + cls];
    for (uint32_t t0 = 0; t0 < nt; t0 += bt)
        for (uint32_t q = 0; q < nch; ++q) {
            const uint32_t s0 = min(src, q * per);
            *it++ = McWork{c, level[c], pt0 + t0, min(bt, nt - t0), s0, min(src, s0 + per) - s0, nch > 1 ? off + q * ((nt + 15) / 16) : ~0u, t0};
        }
}

// Work items of the P2P: counts per leaf, then the plan scalars (items per
// class), written to pinned host words too.  Nothing here waits, so the caller can enqueue other work before
// p2p_run needs the scalars.
void p2p_plan(Ctx &c, bool potential) {
    TreeDev &t = c.t;
    if (!t.nleaves) return;
    const int nl = static_cast<int>(t.nleaves);
    const int nb = static_cast<int>(ceil_div(nl, 256));
    c.p2p_scal.ensure(2 * NCLS + 3);
    c.p2p_nchunk.ensure(nl);
    c.p2p_cls.ensure(nl);
    c.p2p_src.ensure(nl);
    c.p2p_item_off.ensure(nl);
    c.p2p_pre.ensure(static_cast<size_t>(nl) * NSC);
    c.p2p_btot.ensure(static_cast<size_t>(nb) * NBT);
    // under 8 leaves per CU (the 16k Plummer sphere has 430): FP32 items of MC_COST,
    // scaled down by the leaf shortfall, so that there are still several per SIMD;
    // FP64 items take some five times as long, so they shrink from more leaves on
    const int few = (c.prec == 0 ? F64_LEAVES : 8) * c.ncu;
    uint32_t chunk = MC_COST;
    if (nl < few) chunk = std::max<uint32_t>(c.prec == 0 ? F64_MINCOST : MC_MINCOST, static_cast<uint32_t>(1ull * MC_COST * nl / few));
    k_p2p_plan<<<nb, 256, 0, c.stream>>>(t.leaf_ids, nl, t.level, t.count, t.anc, c.p2p_local, c.p2p_nchunk, c.p2p_cls, c.p2p_src, c.p2p_pre, c.p2p_btot, chunk,
                                        c.prec == 0 ? F64_TILES : mc_tiles(potential), nl < 8 * c.ncu ? 1 : 8,
                                        std::max<uint32_t>(PART_ROWS, static_cast<uint32_t>(PART_ENTRIES / c.n)));
    static_assert(2 * NCLS + 3 < 32, "plan scalars");
    k_p2p_plan_blocks<<<1, 256, 0, c.stream>>>(c.p2p_btot, nb, c.p2p_scal, reinterpret_cast<uint32_t *>(static_cast<char *>(c.pinned) + 128), ++c.plan_seq);
    VG_LAUNCH_CHECK();
}

// The plan's scalars, waited for on the host: items per class, class bases,
// tiles of partial sums, split leaves, pieces.
static const uint32_t *p2p_scalars(Ctx &c) {
    const uint32_t *hs = reinterpret_cast<const uint32_t *>(static_cast<const char *>(c.pinned) + 128);
    wait_host_word(hs + 2 * NCLS + 3, c.plan_seq, c.stream);
    return hs;
}

// One launch over all items (one for each piece of the longest), on the stream
// p2p_plan used; L2P adds the partial sums of the leaves split over several.
template <class R>
void p2p_run(Ctx &c, bool potential) {
    using V4 = Quad<R>;
    TreeDev &t = c.t;
    if (!t.nleaves) return;
    const uint32_t *hs = p2p_scalars(c);
    const uint32_t nitems = hs[2 * NCLS - 1] + hs[NCLS - 1], ntiles = hs[2 * NCLS], pieces = hs[2 * NCLS + 2];
    const bool split = hs[2 * NCLS + 1] > 0;
    const int nl = static_cast<int>(t.nleaves);
    c.p2p_items.ensure(sizeof(McWork) * static_cast<size_t>(std::max<uint32_t>(1, nitems)));
    McWork *items = reinterpret_cast<McWork *>(c.p2p_items.p);
    k_p2p_items<<<ceil_div(nl, 256), 256, 0, c.stream>>>(t.leaf_ids, nl, t.level, t.start, t.count, c.p2p_cls, c.p2p_nchunk, c.p2p_src, c.p2p_pre,
                                                         c.p2p_btot, c.p2p_scal, c.p2p_item_off, items, sizeof(R) == 8 ? F64_TILES : mc_tiles(potential));
    VG_LAUNCH_CHECK();
    auto buffers = [&](auto &sorted, auto &sums, auto &parts, auto run) {
        sums.ensure(4 * std::max<int64_t>(1, c.n));
        if (split) parts.ensure(4 * 16 * static_cast<size_t>(ntiles));
        run(reinterpret_cast<const V4 *>(sorted.p), reinterpret_cast<V4 *>(sums.p), reinterpret_cast<V4 *>(parts.p));
    };
    const R G = static_cast<R>(c.G);
    const bool um = !c.has_masses;  // one mass: left out of the pairs, the sums are scaled once
    if constexpr (sizeof(R) == 4) {
        // the units, and what takes sums of m x / r^3 and m / r out of them
        const PairUnits u = PairUnits::of<float>(c);
        const int ls = u.length;
        const double m = um ? c.mass : 1.0;
        const float eps2 = static_cast<float>(u.eps2(c)), unit = static_cast<float>(pow2(-ls));
        const float fscale = static_cast<float>(std::ldexp(m, u.mass - 2 * ls)), pscale = static_cast<float>(std::ldexp(m, u.mass - ls));
        const float m1 = static_cast<float>(pow2(-u.mass));
        bool big = false;  // a root box so wide that squared distances may leave the FP32 range all the same
        for (int a = 0; a < 3; ++a) big |= !((t.box[3 + a] - t.box[a]) * pow2(-ls) < 1e18);
        buffers(c.xs32, c.as32, c.p2p_part32, [&](const V4 *xs, V4 *acc, V4 *part) {
            for (uint32_t p = 0; p < pieces; ++p)
                (potential ? k_p2p_mc<true> : k_p2p_mc<false>)<<<nitems, 64, 0, c.stream>>>(items, t.start, t.count, t.anc, t.ni, t.ni_cnt, t.bmin, t.bmax, xs,
                                                                                       eps2, G, um, m1, big, fscale, pscale, acc, part, unit, p);
        });
    } else {
        const double eps2 = PairUnits::of<double>(c).eps2(c), mu = c.mass;
        buffers(c.xs64, c.as64, c.p2p_part64, [&](const V4 *xs, V4 *acc, V4 *part) {
            for (uint32_t p = 0; p < pieces; ++p)
                (potential ? k_p2p_f64<true> : k_p2p_f64<false>)<<<nitems, 64, 0, c.stream>>>(items, t.start, t.count, t.anc, t.ni, t.ni_cnt, xs, eps2, G, um,
                                                                                         mu, acc, part, p);
        });
    }
    VG_LAUNCH_CHECK();
}

}  // namespace

void fmm_p2p_plan(Ctx &c, bool potential) { p2p_plan(c, potential); }

void fmm_p2p_run(Ctx &c, bool potential) {
    if (c.prec == 0)
        p2p_run<double>(c, potential);
    else
        p2p_run<float>(c, potential);
}

void fmm_p2p(Ctx &c, bool potential) {
    fmm_p2p_plan(c, potential);
    fmm_p2p_run(c, potential);
}

}  // namespace vg
