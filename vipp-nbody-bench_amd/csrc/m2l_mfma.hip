// m2l_mfma.hip - M2L, and in split mode M2M and L2L, on the CDNA4 matrix
// cores with split BF16 operands.
//
// The M2L of one target is L~(t) = sum_o T_o M~(s(t, o)) over its (at most
// 189) source offsets o (fmm.hpp:277-304 in the scaled real basis of
// fmm.hip).  A block owns 64 targets of one child octant qt, so that every
// target sees the same 189 offsets in the same order (offsets follow from
// (parent-neighbour offset, source octant, qt) alone).  Per offset the block
// forms T_o (K x K) times the targets' source multipoles (K x 64) on
// v_mfma_f32_16x16x32_bf16, accumulating in FP32 across its offsets.  Every
// block walks the offsets in the same order, so the operators stream through L2
// shared by the blocks of an XCD.
//
// Precision: every M2L operand x is split as hi = bf16(x), lo = bf16(x - hi)
// (16 significant bits together) and a product is formed as
// hi*hi + hi*lo + lo*hi with FP32 accumulation; the dropped lo*lo term and the
// split residuals are ~2^-18 of the product.  T_o is split from its FP64
// value; the multipoles are split by the kernels that form them (P2M and M2M).  M2M and
// L2L use a three-way split (below).
//
// Operand layouts (checked on the device): for v_mfma_f32_16x16x32_bf16 lane l
// holds A[l%16][8(l/16)+e] and B[8(l/16)+e][l%16], e = 0..7, and
// C[4(l/16) + r][l%16], r = 0..3; for v_mfma_f32_32x32x16_bf16 (M2M, L2L)
// A[l%32][8(l/32)+e], B[8(l/32)+e][l%32] and C[8(r/4) + 4(l/32) + r%4][l%32],
// r = 0..15.  Operators are stored in that A order, so a wavefront loads a
// fragment with one 16-byte read per lane.
#include "gravity.hpp"

namespace vg {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr int mt_of(int K) { return (K + 31) / 32; }
__host__ __device__ constexpr int ks_of(int K) { return (K + 15) / 16; }

// FP64 operators (row-major K x K per offset) -> BF16 hi/lo A fragments of
// the M2L: frag[o][16-row tile][32-column k-step][hi, lo][lane][8 columns], lane
// 16 q + r holding row r, columns 8 q .. 8 q + 7 (zero past K).  One block per
// (offset, row tile): the tile's rows are read into LDS (coalesced), then each
// thread writes whole fragment words.
__global__ __launch_bounds__(256) void k_split_ops(const int16_t *__restrict__ sel, const double *__restrict__ op64, int K, __bf16 *__restrict__ frag,
                                                   int NT, int KS) {
    extern __shared__ double tile[];  // 16 rows x (32 KS + 1)
    const int o = sel[16 + blockIdx.x / NT] - 16, rt = blockIdx.x % NT;  // the M2L offsets of the walk only
    const int kc = 32 * KS, W = kc + 1;
    const double *src = op64 + static_cast<int64_t>(16 + o) * K * K;
    for (int i = threadIdx.x; i < 16 * kc; i += 256) {
        const int r = i / kc, col = i % kc, row = rt * 16 + r;
        tile[r * W + col] = (row < K && col < K) ? src[static_cast<int64_t>(row) * K + col] : 0.0;
    }
    __syncthreads();
    const int64_t base = (static_cast<int64_t>(o) * NT + rt) * KS * 128;  // in 8-coefficient vectors
    for (int v = threadIdx.x; v < KS * 128; v += 256) {
        const int ks = v >> 7, h = (v >> 6) & 1, l = v & 63;
        const int r = l & 15, c0 = ks * 32 + (l >> 4) * 8;
        bf16x8 out;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const double x = tile[r * W + c0 + e];
            const __bf16 hv = static_cast<__bf16>(static_cast<float>(x));
            out[e] = h ? static_cast<__bf16>(static_cast<float>(x - static_cast<double>(static_cast<float>(hv)))) : hv;
        }
        reinterpret_cast<bf16x8 *>(frag)[base + v] = out;
    }
}

// Shape of the split M2L at order P: 64 targets (four 16-target tiles) per
// block, its NT 16-row tiles over WR wavefronts (RW each) and the target tiles
// over WC.  128 targets, two by two wavefronts and three wavefronts for NT = 3
// or 11 were slower (fewer blocks per CU, or operators read twice).
template <int P>
struct SplitShape {
    static constexpr int K = (P + 1) * (P + 1), NT = (K + 15) / 16, KS = (K + 31) / 32;
    static constexpr int TB = 64, WR = NT == 1 ? 1 : NT == 2 ? 2 : 4, WC = 4 / WR;
    static constexpr int RW = (NT + WR - 1) / WR, NC = TB / 16 / WC, NW = WR * WC;
    static constexpr int LD = 16 * ks_of(K);      // coefficients of a cell's row, hi or lo
    static constexpr int CH = LD / 4;             // 16-byte words of a cell's hi and lo rows
    static constexpr int SK = CH | 1;             // the same in LDS: an odd number, so reads have no bank conflicts
    static constexpr int TPI = 64 / CH;           // targets a wavefront gathers with one load
};

// One block: 64 targets (children of octant qt of 64 parents).  Per walked
// offset the block gathers the targets' source multipoles (hi and lo rows, one
// 16-byte word per lane, with this octant's mirror signs) into LDS and
// multiplies the operator by them, hi*hi + hi*lo + lo*hi; operator fragments come
// straight from L2, each loaded by one wavefront where WC = 1, and the next offset's
// multipoles are on their way during the products.  With nsplit > 1 the walked
// offsets are cut into parts, one block each, with partial sums in part.
//
// Bound by the way to L2: at p = 12 a CU takes 26 B/clk of operators and
// multipoles at 47 % of the matrix rate (64 B/clk is its port), so the
// operators are read a k-step ahead (p < 10: four blocks per CU hide the rest;
// two ahead cost a block and 10 to 15 %) or two (p >= 10: two blocks whatever the
// depth; 1 to 3 % faster).  Wavefronts in their products go before the ones that
// gather (s_setprio: -2 % at p = 12).  ms per evaluation, against 32x32x16
// tiles over 32 or 64 targets staged by twice the wavefronts, uncut:
//   Plummer N, p       2461, 4  16384, 8  262144, 8  1M, 9  4M, 8  4M, 10  4M, 12
//   before                .254      .365       .451    .54   1.38    1.75    3.11
//   here                  .026      .058       .095    .38   1.01    1.65    3.13
// and 12.1 -> 11.8 at p = 12 on 16M bodies of two colliding spheres.
template <int P>
__global__ __launch_bounds__(64 * SplitShape<P>::NW, 2) void k_m2l_split(const int32_t *__restrict__ parents, int nparents,
                                                                         const int32_t *__restrict__ child, const uint32_t *__restrict__ count,
                                                                         const int32_t *__restrict__ nbr27, const uint4 *__restrict__ Ms,
                                                                         float *__restrict__ L, const bf16x8 *__restrict__ ops, int nsplit,
                                                                         float *__restrict__ part) {
    using S = SplitShape<P>;
    constexpr int TB = S::TB, NTH = 64 * S::NW;
    constexpr int NG = (TB + S::NW * S::TPI - 1) / (S::NW * S::TPI);  // words a lane gathers
    constexpr int PAD = 4 * S::KS > S::LD / 8 ? 4 * S::KS - S::LD / 8 : 0;  // words read past a row's end (times zero columns)
    __shared__ uint4 sM[TB * S::SK + PAD];
    __shared__ int32_t s_nc[27 * TB];  // first child of parent neighbour d of target t, or -1
    __shared__ uint8_t s_nm[27 * TB];  // its non-empty children
    __shared__ int32_t tgt[TB];
    __shared__ int16_t s_o[189], s_dn[189], s_qs[189], s_live[189];
    __shared__ int s_nlive, s_cnt[3], s_step[189];  // s_step: the walked offsets, operator | neighbour << 9 | octant << 14
    static_assert(NTH >= 192, "m2l_live_steps");
    // XCD-aware placement: blocks go round-robin to the 8 XCDs, so XCD x takes
    // the contiguous run of work items [x W / 8, (x + 1) W / 8); the octant blocks
    // of a parent chunk, which read the same multipoles, share its L2.
    const int nchunks = (nparents + TB - 1) / TB;
    const int per = nchunks * nsplit;
    const int wi = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (wi >= 8 * per) return;
    const int sp = wi % nsplit, w = wi / nsplit, chunk = w >> 3, qt = w & 7;
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, quad = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = (wv + static_cast<int>(blockIdx.x >> 3)) % S::WR, wc = wv / S::WR;  // the light wavefront changes its SIMD from block to block
    m2l_walk(tid, NTH, qt, s_o, s_dn, s_qs);
    if (tid < TB) {
        const int pi = chunk * TB + tid;
        const int32_t p = pi < nparents ? parents[pi] : -1;
        int32_t t = p >= 0 ? child[p] + qt : -1;
        if (t >= 0 && count[t] == 0) t = -1;
        tgt[tid] = t;
        for (int k = S::CH; k < S::SK; ++k) sM[tid * S::SK + k] = make_uint4(0, 0, 0, 0);
    }
    for (int k = tid; k < PAD; k += NTH) sM[TB * S::SK + k] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    for (int i = tid; i < 27 * TB; i += NTH) {
        const int d = i / TB, t = i % TB;
        int32_t cb = -1;
        uint32_t msk = 0;
        if (tgt[t] >= 0) {
            const int32_t p = nbr27[27 * static_cast<int64_t>(parents[chunk * TB + t]) + d];
            cb = p >= 0 ? child[p] : -1;
            if (cb >= 0)
                for (int q = 0; q < 8; ++q) msk |= (count[cb + q] != 0 ? 1u : 0u) << q;
        }
        s_nc[i] = cb;
        s_nm[i] = static_cast<uint8_t>(msk);
    }
    __syncthreads();
    m2l_live_steps(tid, s_live, &s_nlive, s_cnt, [&](int st) {
        const int dn = s_dn[st], qs = s_qs[st];
        int any = 0;
        for (int t = 0; t < TB; ++t) any |= s_nm[dn * TB + t] >> qs;
        return (any & 1) != 0;
    });
    // this lane gathers word ch of the targets (wv + NW u) TPI + sub, with its sign bits (negation commutes with the split)
    const int sub = lane / S::CH, ch = lane % S::CH;
    uint32_t sg[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int k = 8 * (ch % (S::LD / 8)) + 2 * e;
        sg[e] = (k < S::K && m2l_mirror_sign(qt, k) < 0 ? 0x8000u : 0u) | (k + 1 < S::K && m2l_mirror_sign(qt, k + 1) < 0 ? 0x80000000u : 0u);
    }
    const int nlive = s_nlive;
    if (tid < nlive) {
        const int st = s_live[tid];
        s_step[tid] = s_o[st] | s_dn[st] << 9 | s_qs[st] << 14;
    }
    __syncthreads();
    const int lo = sp * nlive / nsplit, hi = (sp + 1) * nlive / nsplit;  // this block's walked offsets
    f32x4 acc[S::RW][S::NC];
#pragma unroll
    for (int r = 0; r < S::RW; ++r)
#pragma unroll
        for (int n = 0; n < S::NC; ++n) acc[r][n] = f32x4{0, 0, 0, 0};
    // fragments of k-step ks of this wavefront's row tiles wr, wr + WR, ... (a missing one repeats the last)
    auto load_a = [&](int li, int ks, bf16x8 (*a)[2]) {
        const bf16x8 *O = ops + static_cast<int64_t>(__builtin_amdgcn_readfirstlane(s_step[li]) & 511) * (S::NT * S::KS * 128) + ks * 128;
#pragma unroll
        for (int r = 0; r < S::RW; ++r) {
            const bf16x8 *F = O + min(wr + S::WR * r, S::NT - 1) * (S::KS * 128);
            a[r][0] = F[static_cast<unsigned>(lane)];
            a[r][1] = F[64u + lane];
        }
    };
    uint4 v[NG];
    uint64_t dead = 0;  // bit u: the target of v[u] has no source here (TPI = 1, which reads row 0 for it)
    static_assert(S::TPI > 1 || S::NW * NG == TB);
    auto gather = [&](int li) {  // this lane's words of the multipoles of walked offset li
        const int st = __builtin_amdgcn_readfirstlane(s_step[li]), dn = (st >> 9 & 31) * TB, qs = st >> 14;
        if constexpr (S::TPI == 1) {  // a load takes one target, whose row lane u has looked up
            const int t = wv + S::NW * (lane % NG);
            const bool live = (s_nm[dn + t] >> qs) & 1;
            const int cell = live ? s_nc[dn + t] + qs : 0;
            dead = ~__ballot(live);
            if (lane < S::CH) {
#pragma unroll
                for (int u = 0; u < NG; ++u) v[u] = (Ms + static_cast<int64_t>(__builtin_amdgcn_readlane(cell, u)) * S::CH)[static_cast<unsigned>(lane)];
            }
            return;
        }
#pragma unroll
        for (int u = 0; u < NG; ++u) {
            v[u] = make_uint4(0, 0, 0, 0);
            const int t = (wv + S::NW * u) * S::TPI + sub;
            if (sub < S::TPI && t < TB && ((s_nm[dn + t] >> qs) & 1)) v[u] = Ms[static_cast<int64_t>(s_nc[dn + t] + qs) * S::CH + ch];
        }
    };
    const uint4 *Brow = sM + (wc * 16 * S::NC + col) * S::SK + quad;
    constexpr int PF = P < 10 ? 1 : 2;  // k-steps of operator in flight (above)
    bf16x8 an[PF][S::RW][2];
    if (hi > lo) {
#pragma unroll
        for (int i = 0; i < PF; ++i) load_a(lo, i, an[i]);
        gather(lo);
    }
    for (int li = lo; li < hi; ++li) {
#pragma unroll
        for (int u = 0; u < NG; ++u) {
            const int t = (wv + S::NW * u) * S::TPI + sub;
            const uint32_t m = S::TPI == 1 && (dead >> u & 1) ? 0u : ~0u;
            if (sub < S::TPI && t < TB) sM[t * S::SK + ch] = make_uint4((v[u].x ^ sg[0]) & m, (v[u].y ^ sg[1]) & m, (v[u].z ^ sg[2]) & m, (v[u].w ^ sg[3]) & m);
        }
        if (li + 1 < hi) gather(li + 1);  // on its way during the products
        __syncthreads();  // the multipoles of this offset are in LDS
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int ks = 0; ks < S::KS; ++ks) {
            bf16x8 a[S::RW][2];
#pragma unroll
            for (int r = 0; r < S::RW; ++r) {
                a[r][0] = an[0][r][0], a[r][1] = an[0][r][1];
#pragma unroll
                for (int i = 0; i + 1 < PF; ++i) an[i][r][0] = an[i + 1][r][0], an[i][r][1] = an[i + 1][r][1];
            }
            if (ks + PF < S::KS)
                load_a(li, ks + PF, an[PF - 1]);
            else if (li + 1 < hi)
                load_a(li + 1, ks + PF - S::KS, an[PF - 1]);
#pragma unroll
            for (int n = 0; n < S::NC; ++n) {
                const bf16x8 bh = __builtin_bit_cast(bf16x8, Brow[16 * n * S::SK + 4 * ks]);
                const bf16x8 bl = __builtin_bit_cast(bf16x8, Brow[16 * n * S::SK + 4 * ks + S::LD / 8]);
#pragma unroll
                for (int r = 0; r < S::RW; ++r) {
                    if (S::NT % S::WR != 0 && r == S::RW - 1 && wr + S::WR * r >= S::NT) continue;
                    acc[r][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r][0], bh, acc[r][n], 0, 0, 0);
                    acc[r][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r][0], bl, acc[r][n], 0, 0, 0);
                    acc[r][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r][1], bh, acc[r][n], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();  // every wavefront has read the multipoles
    }
    // D: lane holds rows 4 quad .. 4 quad + 3 of a tile for target col
#pragma unroll
    for (int r = 0; r < S::RW; ++r) {
        const int tile = wr + S::WR * r, r0 = 16 * tile + 4 * quad;
        if (tile >= S::NT) continue;
#pragma unroll
        for (int n = 0; n < S::NC; ++n) {
            const int ti = (wc * S::NC + n) * 16 + col;
            const int32_t t = tgt[ti];
            if (t < 0) continue;
            f32x4 x = acc[r][n];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (r0 + e < S::K && m2l_mirror_sign(qt, r0 + e) < 0) x[e] = -x[e];
            float *dst = nsplit == 1 ? L + static_cast<int64_t>(t) * S::LD
                                     : part + (static_cast<int64_t>(sp) * 8 * nparents + static_cast<int64_t>(chunk * TB + ti) * 8 + qt) * S::LD;
            *reinterpret_cast<f32x4 *>(dst + r0) = x;
        }
    }
}

// ---------------------------------------------------------------------------
// M2M and L2L of one tree level on the matrix cores.  Their work is small
// (8 operators per level instead of 189 offsets), so they take a three-way
// split, x = h + m + l (BF16 each, 24 significant bits together), and six
// products, hh + hm + mh + hl + mm + lh, which keeps them at FP32 accuracy.
// The 8 M2M (child - parent) and 8 L2L (parent - child) operators are stored
// column-major for the FP32 kernels; their fragments are cut here in the A
// order of the M2L blocks, frag[blk][mt][part][ks][lane][8].
// ---------------------------------------------------------------------------
__device__ __forceinline__ void split3(float x, __bf16 &h, __bf16 &m, __bf16 &l) {
    h = static_cast<__bf16>(x);
    const float r = x - static_cast<float>(h);
    m = static_cast<__bf16>(r);
    l = static_cast<__bf16>(r - static_cast<float>(m));
}

__global__ __launch_bounds__(256) void k_split_ops_ml(const double *__restrict__ op64, int K, __bf16 *__restrict__ frag, int MT, int NKS) {
    const int64_t i = blockIdx.x * 256ll + threadIdx.x;
    const int64_t per = static_cast<int64_t>(MT) * NKS * 64;
    if (i >= 16 * per) return;
    const int blk = static_cast<int>(i / per);
    const int rem = static_cast<int>(i % per);
    const int mt = rem / (NKS * 64), ks = (rem / 64) % NKS, l = rem % 64;
    const double *src = op64 + static_cast<int64_t>(blk) * K * K;
    const int row = mt * 32 + (l & 31);
    const int64_t vec = (static_cast<int64_t>(blk) * MT + mt) * 3 * NKS * 64 + ks * 64 + l;
    for (int e = 0; e < 8; ++e) {
        const int col = ks * 16 + (l >> 5) * 8 + e;
        const double x = (row < K && col < K) ? src[static_cast<int64_t>(col) * K + row] : 0.0;  // column-major
        // the first part from the FP64 value, the other two from the residual
        const __bf16 h = static_cast<__bf16>(static_cast<float>(x));
        __bf16 m, lo, rest;
        split3(static_cast<float>(x - static_cast<double>(static_cast<float>(h))), m, lo, rest);
        frag[vec * 8 + e] = h;
        frag[(vec + NKS * 64) * 8 + e] = m;
        frag[(vec + 2 * NKS * 64) * 8 + e] = lo;
    }
}

// One m-tile of T (fragment block fb) times the expansions src of the lanes' columns (row
// stride 16 NKS; nullptr: zeros): the six products of the three-way split down to 2^-16
// relative, smallest first.  Each lane splits the 8 coefficients that its operand
// holds; those from K on are taken as zero whatever the buffer holds there (the
// locals' padding is not defined).
template <int K>
__device__ __forceinline__ f32x16 ml_tile(const bf16x8 *__restrict__ fb, int mt, int lane, const float *__restrict__ src) {
    constexpr int NKS = ks_of(K);
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const bf16x8 *A = fb + static_cast<size_t>(mt * 3) * NKS * 64 + lane;
    const int half = lane >> 5;
#pragma unroll 4
    for (int ks = 0; ks < NKS; ++ks) {
        const bf16x8 ah = A[ks * 64], am = A[(NKS + ks) * 64], al = A[(2 * NKS + ks) * 64];
        float4 x = make_float4(0, 0, 0, 0), y = x;
        if (src) {
            const float4 *w = reinterpret_cast<const float4 *>(src + 16 * ks + 8 * half);
            x = w[0];
            y = w[1];
        }
        const float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
        bf16x8 bh, bm, bl;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            __bf16 h, m, l;
            split3(16 * ks + 8 * half + e < K ? v[e] : 0.0f, h, m, l);
            bh[e] = h;
            bm[e] = m;
            bl[e] = l;
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am, bm, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bm, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am, bh, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, acc, 0, 0, 0);
    }
    return acc;
}

// M2M (UP, solver_ref.hpp:196-197) and L2L (solver_ref.hpp:217-218) of one level: block =
// (32 parents, one 32-row m-tile), a wavefront each octant q.  M2M: T_q M(child q), zero for
// an empty child, summed in octant order through LDS into the parent's multipoles and
// their halves for M2L.  L2L: L(child q) += T'_q L(parent) for every non-empty child.
// Levels are small, and bound by launches and the latency of one pass; operands come from L2
// straight into registers.  A block per octant, with the expansions split and the result
// put together in LDS, needed a second kernel for the sum over the octants: M2M and L2L per
// evaluation of 100k bodies p = 8 47 + 49 -> 37 + 41 us, L2L of 4M p = 12 226 -> 148, of 16M
// 641 -> 383; a step of 4M 35.96 -> 35.64 ms, closure step of 1M 10.76 -> 10.58 (both with the
// multipoles' halves written here and by P2M, not by a pass of their own).
template <int P, bool UP>
__global__ __launch_bounds__(512) void k_ml_split(const int32_t *__restrict__ ids, int n, const int32_t *__restrict__ child,
                                                  const uint32_t *__restrict__ count, const bf16x8 *__restrict__ frag, float *__restrict__ X, int ldk,
                                                  uint16_t *__restrict__ Ms) {
    constexpr int K = (P + 1) * (P + 1), MT = mt_of(K), NKS = ks_of(K);
    const int lane = threadIdx.x & 63, half = lane >> 5;
    const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int mt = blockIdx.x % MT, i = static_cast<int>(blockIdx.x / MT) * 32 + (lane & 31);
    const int32_t par = i < n ? ids[i] : -1;
    int32_t cell = par >= 0 ? child[par] + q : -1;
    if (cell >= 0 && count[cell] == 0) cell = -1;
    const int32_t from = UP || cell < 0 ? cell : par;
    const f32x16 acc = ml_tile<K>(frag + static_cast<size_t>(UP ? q : 8 + q) * MT * 3 * NKS * 64, mt, lane,
                                  from >= 0 ? X + static_cast<size_t>(from) * ldk : nullptr);
    // acc[4 g + e]: row 32 mt + 8 g + 4 half + e of column lane % 32
    if constexpr (UP) {
        __shared__ f32x4 s_acc[8][4][64];
#pragma unroll
        for (int g = 0; g < 4; ++g) s_acc[q][g][lane] = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
        __syncthreads();
        const int row = 32 * mt + 8 * q + 4 * half;
        if (q < 4 && par >= 0 && row < ldk) {  // wavefront g adds the octants' rows of group g
            f32x4 sum = s_acc[0][q][lane];
#pragma unroll
            for (int o = 1; o < 8; ++o) sum += s_acc[o][q][lane];
            *reinterpret_cast<f32x4 *>(X + static_cast<size_t>(par) * ldk + row) = sum;
            uint32_t h[4], l[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) split_m(sum[e], h[e], l[e]);
            uint16_t *m = Ms + static_cast<size_t>(par) * 2 * ldk + row;
            *reinterpret_cast<uint2 *>(m) = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
            *reinterpret_cast<uint2 *>(m + ldk) = make_uint2(l[0] | l[1] << 16, l[2] | l[3] << 16);
        }
    } else {
        if (cell < 0) return;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int row = 32 * mt + 8 * g + 4 * half;
            if (row < ldk) *reinterpret_cast<f32x4 *>(X + static_cast<size_t>(cell) * ldk + row) += f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
        }
    }
}

template <int P>
void launch_ml(Ctx &c, const int32_t *ids, int64_t n, bool m2m) {
    constexpr int K = (P + 1) * (P + 1);
    const unsigned grid = static_cast<unsigned>(ceil_div(n, 32));
    const bf16x8 *frag = reinterpret_cast<const bf16x8 *>(c.opsplit_ml.p);
    const int np = static_cast<int>(n);
    if (m2m)
        k_ml_split<P, true><<<grid * mt_of(K), 512, 0, c.stream>>>(ids, np, c.t.child, c.t.count, frag, c.M32, c.ldk, c.msplit);
    else
        k_ml_split<P, false><<<grid * mt_of(K), 512, 0, c.stream>>>(ids, np, c.t.child, c.t.count, frag, c.L32, c.ldk, nullptr);
    VG_LAUNCH_CHECK();
}

template <int P>
void launch_split(Ctx &c, const int32_t *parents, int np) {
    using S = SplitShape<P>;
    if (c.ldk != S::LD) throw Error(1, "split M2L: the coefficient stride must be K rounded up to 16");
    const unsigned grid = 8 * ceil_div(np, S::TB);  // one block per (parent chunk, child octant)
    const int nsplit = m2l_parts(grid, c.ncu);
    float *part = m2l_part_sums(c, np, nsplit);
    k_m2l_split<P><<<grid * nsplit, 64 * S::NW, 0, c.stream>>>(parents, np, c.t.child, c.t.count, c.t.nbr27, reinterpret_cast<const uint4 *>(c.msplit.p),
                                                             c.L32, reinterpret_cast<const bf16x8 *>(c.opsplit.p), nsplit, part);
    VG_LAUNCH_CHECK();
    m2l_add_parts(c, parents, np, nsplit, part);
}

}  // namespace

void m2l_split_operators(Ctx &c) {
    const int MT = mt_of(c.K), NKS = ks_of(c.K), NT = ks_of(c.K), KS = mt_of(c.K);  // (16-row tiles, 32-column steps)
    const int64_t per = static_cast<int64_t>(MT) * NKS * 64;
    c.opsplit.ensure(static_cast<size_t>(343) * NT * KS * 128 * 8);
    // split mode runs M2M, M2L and L2L from the fragments: no FP32 copies
    k_split_ops<<<189 * NT, 256, 16 * (32 * KS + 1) * sizeof(double), c.stream>>>(c.ops_sel, c.op64, c.K, reinterpret_cast<__bf16 *>(c.opsplit.p), NT, KS);
    c.opsplit_ml.ensure(static_cast<size_t>(16 * 3 * per * 8));
    k_split_ops_ml<<<ceil_div(16 * per, 256), 256, 0, c.stream>>>(c.op64, c.K, reinterpret_cast<__bf16 *>(c.opsplit_ml.p), MT, NKS);
    VG_LAUNCH_CHECK();
}

void ml_split_level(Ctx &c, const int32_t *ids, int64_t n, bool m2m) {
    if (n <= 0) return;
    switch (c.p) {
        case 1: launch_ml<1>(c, ids, n, m2m); break;
        case 2: launch_ml<2>(c, ids, n, m2m); break;
        case 3: launch_ml<3>(c, ids, n, m2m); break;
        case 4: launch_ml<4>(c, ids, n, m2m); break;
        case 5: launch_ml<5>(c, ids, n, m2m); break;
        case 6: launch_ml<6>(c, ids, n, m2m); break;
        case 7: launch_ml<7>(c, ids, n, m2m); break;
        case 8: launch_ml<8>(c, ids, n, m2m); break;
        case 9: launch_ml<9>(c, ids, n, m2m); break;
        case 10: launch_ml<10>(c, ids, n, m2m); break;
        case 11: launch_ml<11>(c, ids, n, m2m); break;
        case 12: launch_ml<12>(c, ids, n, m2m); break;
        default: throw Error(1, "split M2M / L2L supports 1 <= p <= 12");
    }
}

void fmm_m2l_split_list(Ctx &c, const int32_t *parents, int np) {
    if (np <= 0) return;
    switch (c.p) {
        case 1: launch_split<1>(c, parents, np); break;
        case 2: launch_split<2>(c, parents, np); break;
        case 3: launch_split<3>(c, parents, np); break;
        case 4: launch_split<4>(c, parents, np); break;
        case 5: launch_split<5>(c, parents, np); break;
        case 6: launch_split<6>(c, parents, np); break;
        case 7: launch_split<7>(c, parents, np); break;
        case 8: launch_split<8>(c, parents, np); break;
        case 9: launch_split<9>(c, parents, np); break;
        case 10: launch_split<10>(c, parents, np); break;
        case 11: launch_split<11>(c, parents, np); break;
        case 12: launch_split<12>(c, parents, np); break;
        default: throw Error(1, "split M2L supports 1 <= p <= 12");
    }
}

void fmm_m2l_split(Ctx &c) {
    TreeDev &t = c.t;
    if (t.depth < 1) return;
    const int64_t a = t.int_off[1], b = t.int_off.back();
    if (b <= a) return;
    fmm_m2l_split_list(c, t.int_ids.p + a, static_cast<int>(b - a));
}

}  // namespace vg
