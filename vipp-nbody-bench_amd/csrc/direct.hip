// direct.hip - FP64 direct-sum accelerations of a subset of particles against
// all N, the force oracle of solver_ref_naive.hpp:103-119:
//   a_i = sum_{j != i} G m_j (x_j - x_i) / (|x_j - x_i|^2 + eps^2)^{3/2}
// (and, on request, the potential sum_{j != i} m_j / sqrt(|x_j - x_i|^2 + eps^2)
// without G).  Used to measure the FMM's force error on large samples.
//
// Layout: one thread per target, the sources streamed through LDS in tiles of
// 256 (x, y, z, m) FP64 records.  The source range is cut into S slices (grid
// y) so that a few thousand targets still fill the chip; the S partial sums of
// a target are added in slice order afterwards, so the result does not depend
// on scheduling.
#include <algorithm>
#include <atomic>
#include <climits>
#include <mutex>

#include "gravity.hpp"

namespace vg {
namespace {

constexpr int DT = 256;  // threads per block and sources per LDS tile

// One source's terms as the reference forms them, for any distance.
template <bool POT>
__device__ inline void add_exact(double dx, double dy, double dz, double Gm, double m, double eps2, double *s) {
    const double r2 = dx * dx + dy * dy + dz * dz + eps2;
    const double r = sqrt(r2);
    const double gm = Gm / (r2 * r);
    s[0] += gm * dx, s[1] += gm * dy, s[2] += gm * dz;
    if (POT) s[3] += m / r;
}

// The same from v_rsq_f64's y (2^-24 at worst): with e = 1 - r2 y^2,
// r2^(-3/2) = y^3 (1 + 3/2 e + 15/8 e^2 + O(e^3)) and 1 / r = y (1 + e / 2 +
// 3/8 e^2 + ..), e^3 below 2^-69.  A correctly rounded square root and quotient
// take three times the instructions.  r2 = 0 and r2 = inf give NaN (see below).
template <bool POT>
__device__ inline void add_fast(double dx, double dy, double dz, double r2, double gm, double m, double *s) {
    const double y = __builtin_amdgcn_rsq(r2);
    const double yy = y * y;
    const double e = fma(-r2, yy, 1.0);
    const double c = (y * gm) * yy;
    const double f = fma(c * e, fma(e, 1.875, 1.5), c);
    s[0] = fma(f, dx, s[0]), s[1] = fma(f, dy, s[1]), s[2] = fma(f, dz, s[2]);
    if (POT) s[3] = fma(m, fma(y * e, fma(e, 0.375, 0.5), y), s[3]);
}

// bad (may be null): set to 1 when a target index lies outside [0, n); such
// a target is skipped (the host-side entry point checks indices beforehand).
//
// Bound by FP64 issue: 16 operations at 4.6 cycles and one v_rsq_f64 (16) for
// 64 pairs.  4096 targets of 1M sources: 6.2 -> 2.9 ms, 65,536 of 100,000: 9.7 ->
// 4.5 ms (sources through scalar loads instead of LDS: 0.3 ms more).  A target of
// its own (solver_ref_naive.hpp:111-113) costs something only in the tiles that
// hold one of the wavefront's targets.  By the reference's operations are formed a
// tile's sum that is not finite (a source at the target's place without softening,
// distances whose square overflows; one such pair, 256 targets of 2^18 sources: 0.37 ->
// 0.39 ms, 1.17 with its thread walking the slice again) and the sums over up to
// EXACT_N sources: callers, the tests among them, compare the forces of tiny systems with
// the formula component by component at 1e-13, and where terms cancel any other
// rounding shows (4.7e-13 at 64 sources).  A call is its launches and copies there (128 of
// 128: 50 us, against 42; 256 of 256: 78 against 51).
constexpr int64_t EXACT_N = 128;
template <bool POT>
__global__ __launch_bounds__(DT) void k_direct(const double *__restrict__ x, const double *__restrict__ masses, double mass, int64_t n,
                                               const int64_t *__restrict__ idx, int64_t nidx, int64_t slice, double G, double eps2,
                                               double *__restrict__ part, double *__restrict__ bad) {
    __shared__ double2 sxy[DT], szg[DT];  // (x, y), (z, G m)
    __shared__ double sm[POT ? DT : 1];
    const int64_t k = blockIdx.x * static_cast<int64_t>(DT) + threadIdx.x;
    const int64_t i0 = k < nidx ? idx[k] : -1;
    const bool live = k < nidx && i0 >= 0 && i0 < n;
    if (k < nidx && !live && bad) *bad = 1.0;
    const int64_t i = live ? i0 : -1;
    const double xi = live ? x[3 * i] : 0, yi = live ? x[3 * i + 1] : 0, zi = live ? x[3 * i + 2] : 0;
    const int64_t j0 = blockIdx.y * slice;
    const int64_t j1 = j0 + slice < n ? j0 + slice : n;
    double s[4] = {0, 0, 0, 0};
    for (int64_t b = j0; b < j1; b += DT) {
        __syncthreads();
        const int64_t j = b + threadIdx.x;
        if (j < j1) {
            const double m = masses ? masses[j] : mass;
            sxy[threadIdx.x] = make_double2(x[3 * j], x[3 * j + 1]);
            szg[threadIdx.x] = make_double2(x[3 * j + 2], G * m);
            if (POT) sm[threadIdx.x] = m;
        }
        __syncthreads();
        const int nt = j1 - b < DT ? static_cast<int>(j1 - b) : DT;
        const int self = i >= b && i < b + nt ? static_cast<int>(i - b) : -1;
        double t[4] = {0, 0, 0, 0};  // the tile's sums
        bool exact = n <= EXACT_N;
        if (!exact) {
            if (__ballot(self >= 0) == 0) {
#pragma unroll 4
                for (int u = 0; u < nt; ++u) {
                    const double dx = sxy[u].x - xi, dy = sxy[u].y - yi, dz = szg[u].x - zi;
                    add_fast<POT>(dx, dy, dz, fma(dx, dx, fma(dy, dy, fma(dz, dz, eps2))), szg[u].y, POT ? sm[u] : 0.0, t);
                }
            } else {
                for (int u = 0; u < nt; ++u) {
                    const double dx = sxy[u].x - xi, dy = sxy[u].y - yi, dz = szg[u].x - zi;
                    const double r2 = u == self ? 1.0 : fma(dx, dx, fma(dy, dy, fma(dz, dz, eps2)));  // adds 0 dx = 0
                    add_fast<POT>(dx, dy, dz, r2, szg[u].y, POT && u != self ? sm[u] : 0.0, t);
                }
            }
            exact = live && !(isfinite(t[0]) && isfinite(t[1]) && isfinite(t[2]) && isfinite(t[3]));
        }
        if (exact) {
            t[0] = t[1] = t[2] = t[3] = 0;
            for (int u = 0; u < nt; ++u)
                if (u != self) add_exact<POT>(sxy[u].x - xi, sxy[u].y - yi, szg[u].x - zi, szg[u].y, POT ? sm[u] : 0.0, eps2, t);
        }
        for (int c = 0; c < 4; ++c) s[c] += t[c];
    }
    if (k >= nidx) return;
    double *o = part + (static_cast<int64_t>(blockIdx.y) * nidx + k) * 4;
    for (int c = 0; c < 4; ++c) o[c] = live ? s[c] : 0.0;
}

__global__ __launch_bounds__(256) void k_direct_sum(const double *__restrict__ part, int64_t nidx, int S, double *__restrict__ a,
                                                    double *__restrict__ pot) {
    const int64_t k = blockIdx.x * 256ll + threadIdx.x;
    if (k >= nidx) return;
    double s[4] = {0, 0, 0, 0};
    for (int y = 0; y < S; ++y)
        for (int c = 0; c < 4; ++c) s[c] += part[(static_cast<int64_t>(y) * nidx + k) * 4 + c];
    a[3 * k] = s[0];
    a[3 * k + 1] = s[1];
    a[3 * k + 2] = s[2];
    if (pot) pot[k] = s[3];
}

__global__ void k_clear(double *__restrict__ w) { *w = 0.0; }

// Scratch of the allocation-free entry point: partial sums of up to
// NOALLOC_RECORDS (target, slice) records of 4 doubles, then one flag word.
// Each device holds its own copy; host code reaches it only through the
// address hipGetSymbolAddress gives for that device (noalloc_scratch()).
constexpr int64_t NOALLOC_RECORDS = int64_t(1) << 19;  // 16 MiB of partial sums
static __device__ __align__(256) double scratch[4 * NOALLOC_RECORDS + 32];

// slices of the source range: enough blocks to fill the chip, each slice at
// least 4096 sources, at most max_records / nidx of them
int64_t direct_slices(int64_t n, int64_t nidx, int64_t max_records) {
    const int64_t tblocks = ceil_div(nidx, DT);
    int64_t S = std::max<int64_t>(1, std::min<int64_t>(ceil_div(4096, tblocks), ceil_div(n, 4096)));
    S = std::min<int64_t>(S, 65535);
    S = std::max<int64_t>(1, std::min<int64_t>(S, max_records / nidx));
    return S;
}

void launch_direct(Ctx &c, const int64_t *idx, int64_t nidx, double *part, int64_t S, double *a, double *pot, double *bad) {
    const int64_t slice = ceil_div(c.n, S);
    S = ceil_div(c.n, slice);
    const dim3 grid(ceil_div(nidx, DT), static_cast<unsigned>(S));
    (pot ? k_direct<true> : k_direct<false>)<<<grid, DT, 0, c.stream>>>(c.x, c.has_masses ? c.m.p : nullptr, c.mass, c.n, idx, nidx, slice, c.G,
                                                                        c.eps * c.eps, part, bad);
    VG_LAUNCH_CHECK();
    k_direct_sum<<<ceil_div(nidx, 256), 256, 0, c.stream>>>(part, nidx, static_cast<int>(S), a, pot);
    VG_LAUNCH_CHECK();
}

// the device address of `scratch` on each device ordinal, set once per device
// by noalloc_init (the array's host-side name is not a device address)
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
std::atomic<double *> g_scratch_ptr[MAX_DEVICES];

}  // namespace

void noalloc_init(int device) {
    if (device < 0 || device >= MAX_DEVICES) throw Error(1, "device ordinal out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device].load()) return;
    int cur = -1;
    VG_HIP(hipGetDevice(&cur));
    if (cur != device) throw Error(4, "noalloc_init: the device must be current");
    void *q = nullptr;
    VG_HIP(hipGetSymbolAddress(&q, HIP_SYMBOL(scratch)));
    g_scratch_ptr[device].store(static_cast<double *>(q));
}

void direct_subset_noalloc(Ctx &c, const int64_t *idx, int64_t nidx, double *a, double *pot) {
    if (nidx <= 0) return;
    if (nidx > NOALLOC_RECORDS) throw Error(1, "direct (no allocation): more than 524288 targets in one call");
    double *scr = c.device >= 0 && c.device < MAX_DEVICES ? g_scratch_ptr[c.device].load() : nullptr;
    if (!scr) throw Error(5, "direct (no allocation): scratch of this device not set up");
    double *bad = scr + 4 * NOALLOC_RECORDS;
    k_clear<<<1, 1, 0, c.stream>>>(bad);
    VG_LAUNCH_CHECK();
    launch_direct(c, idx, nidx, scr, direct_slices(c.n, nidx, NOALLOC_RECORDS), a, pot, bad);
    double *hflag = reinterpret_cast<double *>(static_cast<char *>(c.pinned) + Ctx::PINNED_BYTES - 64);  // a pinned host word
    VG_HIP(hipMemcpyAsync(hflag, bad, sizeof(double), hipMemcpyDeviceToHost, c.stream));
    VG_HIP(hipStreamSynchronize(c.stream));
    if (*hflag != 0.0) throw Error(1, "direct: particle index out of range");
}

void direct_subset(Ctx &c, const int64_t *idx_host, int64_t nidx, double *a_host, double *pot_host) {
    if (nidx <= 0) return;
    for (int64_t k = 0; k < nidx; ++k)
        if (idx_host[k] < 0 || idx_host[k] >= c.n) throw Error(1, "direct: particle index out of range");
    const int64_t S = direct_slices(c.n, nidx, INT64_MAX);
    // partial sums, results and indices: the context's buffers up to KEEP words, since allocating and
    // freeing them took 50 to 110 us a call (4096 targets of 1M: 3.00 -> 2.89 ms); larger ones are freed on return
    constexpr size_t KEEP = 1 << 23;
    const size_t npart = static_cast<size_t>(S) * nidx * 4, words = npart + 4 * static_cast<size_t>(nidx);
    DevBuf<int64_t> own_idx;
    DevBuf<double> own_buf;
    DevBuf<int64_t> &idx = words <= KEEP ? c.dir_idx : own_idx;
    DevBuf<double> &buf = words <= KEEP ? c.dir_buf : own_buf;
    idx.ensure(nidx);
    buf.ensure(words);
    double *part = buf.p, *a = part + npart, *pot = pot_host ? a + 3 * nidx : nullptr;
    VG_HIP(hipMemcpyAsync(idx.p, idx_host, nidx * sizeof(int64_t), hipMemcpyHostToDevice, c.stream));
    launch_direct(c, idx, nidx, part, S, a, pot, nullptr);
    VG_HIP(hipMemcpyAsync(a_host, a, 3 * nidx * sizeof(double), hipMemcpyDeviceToHost, c.stream));
    if (pot) VG_HIP(hipMemcpyAsync(pot_host, pot, nidx * sizeof(double), hipMemcpyDeviceToHost, c.stream));
    VG_HIP(hipStreamSynchronize(c.stream));  // the caller's arrays are filled; own buffers are released on return
}

}  // namespace vg
