// sort.hip - stable LSD radix sort of (u64 key, u32 value) pairs.
//
// Three kernels per digit of up to 9 bits (the passes split the key bits
// evenly: 36 bits take 4 passes of 9, 64 take 8 of 8): a tile histogram, a
// per-digit scan over the tiles (which also gives each digit's total; left to the
// scatter where the tiles are few), and a scatter that ranks equal digits with ballots, wavefront by wavefront in key
// order, so the order of equal keys is kept (the tree needs points of a cell
// in the caller's index order).  The scatter reorders each tile in LDS before
// writing, so its global writes are runs of consecutive addresses.
#include "gravity.hpp"

namespace vg {
namespace {

constexpr int RS_THREADS = 512;
constexpr int RS_ITEMS = 8;
constexpr int RS_TILE = RS_THREADS * RS_ITEMS;
constexpr int RS_MAXBITS = 9;
constexpr int RS_BINS = 1 << RS_MAXBITS;  // bins held; a pass of b bits uses the first 2^b
constexpr int RS_BPT = RS_BINS / RS_THREADS;
constexpr int RS_WAVES = RS_THREADS / 64;
static_assert(RS_BINS % RS_THREADS == 0, "whole bins per thread");
// Launches bound the small sorts, so up to one tile is sorted by one kernel (500
// particles: an evaluation of 240 -> 219 us, 4096: 309 -> 280 us) and up to RS_FEW
// tiles do without the scan (16384: 409 -> 396 us, 2^18: 907 -> 900 us; with a bound
// of 256 tiles the sums in every block cost more than the scan: 2^20 1650 -> 1690 us).
constexpr unsigned RS_FEW = 64;

// hist[bin][tile], or for the scatter that scans by itself (FEW) hist[tile][bin]
template <bool FEW>
__global__ __launch_bounds__(RS_THREADS) void k_rs_hist(const uint64_t *__restrict__ key, int64_t n, int shift, unsigned mask, uint32_t *__restrict__ hist,
                                                        unsigned ntiles) {
    __shared__ uint32_t h[RS_BINS];
    const unsigned tile = blockIdx.x;
#pragma unroll
    for (int q = 0; q < RS_BPT; ++q) h[threadIdx.x + q * RS_THREADS] = 0;
    __syncthreads();
    const int64_t base = static_cast<int64_t>(tile) * RS_TILE;
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r) {
        const int64_t i = base + r * RS_THREADS + threadIdx.x;
        if (i < n) atomicAdd(&h[(key[i] >> shift) & mask], 1u);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RS_BPT; ++q) {
        const unsigned b = threadIdx.x + q * RS_THREADS;
        if (b > mask) break;
        hist[FEW ? static_cast<size_t>(tile) * (mask + 1) + b : static_cast<size_t>(b) * ntiles + tile] = h[b];
    }
}

// one block per digit value: exclusive scan of hist[bin][0..ntiles) in
// place, and the digit's total into bin_total[bin]
__global__ __launch_bounds__(1024) void k_rs_scan(uint32_t *__restrict__ hist, uint32_t *__restrict__ bin_total, unsigned ntiles) {
    __shared__ uint32_t warp_sum[16];
    __shared__ uint32_t carry;
    const unsigned bin = blockIdx.x;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    uint32_t *row = hist + static_cast<size_t>(bin) * ntiles;
    for (unsigned off = 0; off < ntiles; off += 1024) {
        const unsigned i = off + threadIdx.x;
        const uint32_t v = i < ntiles ? row[i] : 0u;
        // inclusive scan within the wavefront
        uint32_t s = v;
        const unsigned lane = threadIdx.x & 63;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(s, d, 64);
            if (lane >= static_cast<unsigned>(d)) s += o;
        }
        if (lane == 63) warp_sum[threadIdx.x >> 6] = s;
        __syncthreads();
        uint32_t wbase = 0;
        for (unsigned w = 0; w < (threadIdx.x >> 6); ++w) wbase += warp_sum[w];
        const uint32_t c0 = carry;
        if (i < ntiles) row[i] = c0 + wbase + s - v;
        __syncthreads();
        if (threadIdx.x == 1023) carry = c0 + wbase + s;
        __syncthreads();
    }
    if (threadIdx.x == 0) bin_total[bin] = carry;
}

// exclusive scan of one value per thread over the block (RS_THREADS threads)
__device__ inline uint32_t block_excl_scan(uint32_t v, uint32_t *wsum, uint32_t &total) {
    const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(x, d, 64);
        if (lane >= static_cast<unsigned>(d)) x += o;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    uint32_t wb = 0, t = 0;
#pragma unroll
    for (int w = 0; w < RS_WAVES; ++w) {
        wb += static_cast<unsigned>(w) < wave ? wsum[w] : 0u;
        t += wsum[w];
    }
    total = t;
    return wb + x - v;
}

// One 4096-key tile in LDS (512 threads x 8 keys).
struct RsTile {
    uint64_t k[RS_TILE];
    uint32_t v[RS_TILE];
    uint32_t wc[RS_WAVES][RS_BINS];  // keys per (wavefront, digit); then the wavefront's tile-local start
    uint32_t start[RS_BINS];         // tile-local start of each digit
    uint32_t wsum[RS_WAVES];
};

// Reorders the tile by one digit: key r of a thread is key
// 512 wave + 64 r + lane of the tile's nt, in its registers on entry, and all
// are in S.k, S.v in the new order on return (a barrier before they are read).
// Wavefront w ranks the contiguous keys [512 w, 512 w + 512) of the tile in 8
// rounds of 64, in order: the lanes with equal digits find each other with
// ballots, and a running count per (wavefront, digit) gives each key its rank
// among the wavefront's keys of that digit, so equal keys keep their order.  One
// block scan then turns the per-wavefront counts into tile-local starts.
__device__ __forceinline__ void rs_reorder(RsTile &S, int nt, int shift, int bits, const uint64_t (&k)[RS_ITEMS], const uint32_t (&v)[RS_ITEMS]) {
    static_assert(RS_BINS == RS_THREADS, "one digit per thread in the scans");
    static_assert(RS_TILE == RS_WAVES * RS_ITEMS * 64, "each wavefront ranks RS_ITEMS rounds of 64 keys");
    const unsigned mask = (1u << bits) - 1u;
    const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int j0 = static_cast<int>(wave * (RS_ITEMS * 64) + lane);
#pragma unroll
    for (int w = 0; w < RS_WAVES; ++w) S.wc[w][threadIdx.x] = 0;
    __syncthreads();
    uint32_t lp[RS_ITEMS];
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r) {
        const bool ok = j0 + r * 64 < nt;
        const unsigned d = static_cast<unsigned>((k[r] >> shift) & mask);
        uint64_t match = __ballot(ok);
        for (int b = 0; b < bits; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bal = __ballot(bit);
            match &= bit ? bal : ~bal;
        }
        const unsigned rank = __popcll(match & lt);
        const unsigned cnt = __popcll(match);
        const uint32_t c0 = ok ? S.wc[wave][d] : 0u;  // read by every lane of the digit before its last lane updates it
        lp[r] = c0 + rank;
        if (ok && rank == cnt - 1) S.wc[wave][d] = c0 + cnt;
    }
    __syncthreads();
    {
        const unsigned b = threadIdx.x;  // digit
        uint32_t run = 0;
#pragma unroll
        for (int w = 0; w < RS_WAVES; ++w) {
            const uint32_t c = S.wc[w][b];
            S.wc[w][b] = run;
            run += c;
        }
        uint32_t tot;
        const uint32_t st = block_excl_scan(run, S.wsum, tot);  // tile-local start of digit b
        S.start[b] = st;
#pragma unroll
        for (int w = 0; w < RS_WAVES; ++w) S.wc[w][b] += st;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r)
        if (j0 + r * 64 < nt) {
            const unsigned d = static_cast<unsigned>((k[r] >> shift) & mask);
            const uint32_t pos = S.wc[wave][d] + lp[r];
            S.k[pos] = k[r];
            S.v[pos] = v[r];
        }
}

// Scatter of one tile: reordered in LDS and written out in that order, so
// consecutive threads write consecutive addresses of each digit's run.  hist holds
// the tile's start within each digit (exclusive over tiles), bin_total each
// digit's total, whose exclusive scan is the digit's start in the output; with
// FEW hist holds the tiles' own counts, and each block adds up those before it
// and all.
template <bool FEW>
__global__ __launch_bounds__(RS_THREADS) void k_rs_scatter(const uint64_t *__restrict__ key, const uint32_t *__restrict__ val, uint64_t *__restrict__ key_out,
                                                           uint32_t *__restrict__ val_out, int64_t n, int shift, int bits,
                                                           const uint32_t *__restrict__ hist, const uint32_t *__restrict__ bin_total, unsigned ntiles) {
    __shared__ RsTile S;
    __shared__ uint32_t gbase[RS_BINS];  // output position of each digit's first key of this tile
    const unsigned mask = (1u << bits) - 1u;
    const unsigned tile = blockIdx.x;
    const int64_t base = static_cast<int64_t>(tile) * RS_TILE;
    const int nt = static_cast<int>(min<int64_t>(RS_TILE, n - base));
    const int j0 = static_cast<int>((threadIdx.x >> 6) * (RS_ITEMS * 64) + (threadIdx.x & 63));
    uint64_t k[RS_ITEMS];
    uint32_t v[RS_ITEMS];
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r) {
        const bool ok = j0 + r * 64 < nt;
        k[r] = ok ? key[base + j0 + r * 64] : 0ull;
        v[r] = ok ? val[base + j0 + r * 64] : 0u;
    }
    const unsigned b = threadIdx.x;  // digit
    uint32_t bt = 0, before = 0;
    if (b <= mask) {
        if (FEW) {
#pragma unroll 8
            for (unsigned u = 0; u < ntiles; ++u) {
                const uint32_t c = hist[static_cast<size_t>(u) * (mask + 1) + b];
                before += u < tile ? c : 0u;
                bt += c;
            }
        } else {
            bt = bin_total[b];
            before = hist[static_cast<size_t>(b) * ntiles + tile];
        }
    }
    rs_reorder(S, nt, shift, bits, k, v);
    __syncthreads();  // wsum is used again; the tile is whole
    uint32_t tot;
    gbase[b] = block_excl_scan(bt, S.wsum, tot) + before;  // output start of digit b
    __syncthreads();
    // write out in LDS order: slot j of digit d goes to its output run
    for (int j = threadIdx.x; j < nt; j += RS_THREADS) {
        const uint64_t kk = S.k[j];
        const unsigned d = static_cast<unsigned>((kk >> shift) & mask);
        const uint32_t pos = gbase[d] + (j - S.start[d]);
        key_out[pos] = kk;
        val_out[pos] = S.v[j];
    }
}

// All passes of up to one tile, in LDS.
__global__ __launch_bounds__(RS_THREADS) void k_rs_tile(uint64_t *__restrict__ key, uint32_t *__restrict__ val, int n, int begin_bit, int end_bit, int width) {
    __shared__ RsTile S;
    const int j0 = static_cast<int>((threadIdx.x >> 6) * (RS_ITEMS * 64) + (threadIdx.x & 63));
    uint64_t k[RS_ITEMS];
    uint32_t v[RS_ITEMS];
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r) {
        const bool ok = j0 + r * 64 < n;
        k[r] = ok ? key[j0 + r * 64] : 0ull;
        v[r] = ok ? val[j0 + r * 64] : 0u;
    }
    for (int shift = begin_bit; shift < end_bit; shift += width) {
        rs_reorder(S, n, shift, min(width, end_bit - shift), k, v);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < RS_ITEMS; ++r)
            if (j0 + r * 64 < n) {
                k[r] = S.k[j0 + r * 64];
                v[r] = S.v[j0 + r * 64];
            }
    }
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r)
        if (j0 + r * 64 < n) {
            key[j0 + r * 64] = k[r];
            val[j0 + r * 64] = v[r];
        }
}

}  // namespace

// Sorts (k, v) by bits [begin_bit, end_bit) of k; on return k/v point to the
// sorted data (the buffers may have been swapped with k_alt/v_alt).
void radix_sort_pairs(hipStream_t st, uint64_t *&k, uint32_t *&v, uint64_t *&k_alt, uint32_t *&v_alt, int64_t n, int begin_bit, int end_bit,
                      DevBuf<uint32_t> &hist) {
    if (n <= 1) return;
    const unsigned ntiles = ceil_div(static_cast<size_t>(n), RS_TILE);
    hist.ensure(static_cast<size_t>(RS_BINS) * ntiles + RS_BINS);
    uint32_t *bin_total = hist.p + static_cast<size_t>(RS_BINS) * ntiles;
    const int nbits = end_bit - begin_bit;
    const int passes = (nbits + RS_MAXBITS - 1) / RS_MAXBITS;
    const int width = (nbits + passes - 1) / passes;  // <= RS_MAXBITS
    if (ntiles == 1) {
        k_rs_tile<<<1, RS_THREADS, 0, st>>>(k, v, static_cast<int>(n), begin_bit, end_bit, width);
        VG_LAUNCH_CHECK();
        return;
    }
    for (int shift = begin_bit; shift < end_bit; shift += width) {
        const int bits = std::min(width, end_bit - shift);
        const unsigned nbins = 1u << bits;
        if (ntiles <= RS_FEW) {
            k_rs_hist<true><<<ntiles, RS_THREADS, 0, st>>>(k, n, shift, nbins - 1, hist.p, ntiles);
            k_rs_scatter<true><<<ntiles, RS_THREADS, 0, st>>>(k, v, k_alt, v_alt, n, shift, bits, hist.p, nullptr, ntiles);
        } else {
            k_rs_hist<false><<<ntiles, RS_THREADS, 0, st>>>(k, n, shift, nbins - 1, hist.p, ntiles);
            k_rs_scan<<<nbins, 1024, 0, st>>>(hist.p, bin_total, ntiles);
            k_rs_scatter<false><<<ntiles, RS_THREADS, 0, st>>>(k, v, k_alt, v_alt, n, shift, bits, hist.p, bin_total, ntiles);
        }
        VG_LAUNCH_CHECK();
        std::swap(k, k_alt);
        std::swap(v, v_alt);
    }
}

}  // namespace vg
