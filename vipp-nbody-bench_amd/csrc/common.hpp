// common.hpp - shared definitions of the MI355X gravity FMM library.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

namespace vg {

// 21 octal digits fit one 63-bit path code; a tree deeper than that is refused.
constexpr int MAXD = 21;
// Expansion order limit: (p+1)^2 <= 169 real coefficients per cell.
constexpr int MAXP = 12;
constexpr int MAXK = (MAXP + 1) * (MAXP + 1);
// Operators built per evaluation: 8 M2M, 8 L2L and the 189 M2L offsets of
// octant 0's walk (m2l_step below; the other octants reuse them mirrored).
constexpr int NOPS_USED = 16 + 189;

struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

#define VG_HIP(expr)                                                                                              \
    do {                                                                                                          \
        hipError_t _e = (expr);                                                                                   \
        if (_e != hipSuccess)                                                                                     \
            throw ::vg::Error(4, std::string("HIP error ") + hipGetErrorString(_e) + " at " + __FILE__ + ":" +  \
                                     std::to_string(__LINE__) + " (" #expr ")");                                 \
    } while (0)

#define VG_LAUNCH_CHECK() VG_HIP(hipGetLastError())

inline unsigned ceil_div(size_t a, size_t b) { return static_cast<unsigned>((a + b - 1) / b); }

// Device buffer that can grow; grow() keeps the old contents when asked.
template <class T>
struct DevBuf {
    T *p = nullptr;
    size_t cap = 0;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() { release(); }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        cap = 0;
    }
    void ensure(size_t n, bool keep = false, hipStream_t st = nullptr) {
        if (n <= cap) return;
        size_t nc = cap ? cap : 1024;
        while (nc < n) nc *= 2;
        T *q = nullptr;
        VG_HIP(hipMalloc(&q, nc * sizeof(T)));
        if (keep && p && cap) VG_HIP(hipMemcpyAsync(q, p, cap * sizeof(T), hipMemcpyDeviceToDevice, st));
        if (p) {
            if (keep) VG_HIP(hipStreamSynchronize(st));
            (void)hipFree(p);
        }
        p = q;
        cap = nc;
    }
    void swap(DevBuf &o) noexcept {
        std::swap(p, o.p);
        std::swap(cap, o.cap);
    }
    operator T *() const { return p; }
};

// Four values of a particle in one 16- or 32-byte word.
template <class R>
struct QuadOf;
template <>
struct QuadOf<float> {
    using T = float4;
};
template <>
struct QuadOf<double> {
    using T = double4;
};
template <class R>
using Quad = typename QuadOf<R>::T;

__device__ inline float rsq(float x) { return __builtin_amdgcn_rsqf(x); }

// The FP32 near field forms masses times positions and r^-3 by themselves, so it
// takes positions in units of 2^length_shift and masses in units of 2^mass_shift, which
// its last factors undo: powers of two, so no rounding changes, and 1 in ordinary
// units.  Lengths to 2^40 need none (r^-3 above 2^-123, normal); a root box wider
// than 2^64, whose squares FP32 does not hold, is shifted as one of 2^64, so that
// clusters small beside it keep their range; a softening of any size is shifted in
// full, since nothing counts beside it.  Masses to 2^40 need none, larger ones are taken
// to 2^40 (times 2^41: 2^81); and where shorter lengths would make m / eps^3, which the pair
// of a particle with itself forms and multiplies by 0, leave the range, masses are
// shifted by up to three times as much, so that it is no larger than in the caller's units.
__host__ __device__ inline int exponent_of(double v) {  // |v| < 2^e, at least half of that
    return static_cast<int>(__builtin_bit_cast(uint64_t, v) >> 52 & 0x7ff) - 1022;
}
__host__ __device__ inline double pow2(int e) { return __builtin_bit_cast(double, static_cast<uint64_t>(1023 + e) << 52); }  // -1022 <= e <= 1023
__host__ __device__ inline int length_shift(const double *box, double eps) {
    int e = exponent_of(fmax(fmax(box[3] - box[0], box[4] - box[1]), box[5] - box[2]));
    if (e > 64) e = 64;
    if (exponent_of(eps) > e) e = exponent_of(eps);
    return e > 40 ? e - 40 : 0;
}
__host__ __device__ inline int mass_shift(int length, double largest, double eps) {
    const int em = exponent_of(largest);
    int b = em > 40 ? em - 40 : 0;
    if (eps != 0) {
        const int self = em + 3 * (length + 1 - exponent_of(eps)) - 126, most = 3 * length;  // m / eps^3 below 2^126
        const int need = self < most ? self : most;
        if (need > b) b = need;
    }
    return b;
}

// x as two BF16 halves, hi = bf16(x) and lo = bf16(x - hi) (the split M2L's multipoles).
__device__ __forceinline__ void split_m(float x, uint32_t &hi, uint32_t &lo) {
    const __bf16 h = static_cast<__bf16>(x);
    hi = __builtin_bit_cast(uint16_t, h);
    lo = __builtin_bit_cast(uint16_t, static_cast<__bf16>(x - static_cast<float>(h)));
}

// Real-packed index of a degree-n, order-m (m >= 0) coefficient: degree n owns
// entries [n*n, (n+1)*(n+1)): Re(m=0), then (Re, Im) for m = 1..n.
__host__ __device__ inline int kidx_re(int n, int m) { return m == 0 ? n * n : n * n + 2 * m - 1; }
__host__ __device__ inline int kidx_im(int n, int m) { return n * n + 2 * m; }

// Block-wide minimum and maximum of each coordinate and a non-finite flag
// over a block of 256 threads, stored as the 7 doubles of one partial box
// (lo xyz, hi xyz, flag) at part.  Every thread of the block must call it.
__device__ inline void aabb_block_store(const double *lo, const double *hi, double bad, double *part) {
    __shared__ double s[7][256];
    for (int a = 0; a < 3; ++a) {
        s[a][threadIdx.x] = lo[a];
        s[3 + a][threadIdx.x] = hi[a];
    }
    s[6][threadIdx.x] = bad;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < static_cast<unsigned>(w))
            for (int a = 0; a < 7; ++a)
                s[a][threadIdx.x] = a < 3 ? fmin(s[a][threadIdx.x], s[a][threadIdx.x + w]) : fmax(s[a][threadIdx.x], s[a][threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x < 7) part[threadIdx.x] = s[threadIdx.x][0];
}

// M2L by mirror symmetry.  The 189 well-separated (parent neighbour d, source
// octant q) pairs of a target of octant 0 are walked in one fixed order; for a
// target of octant qt the geometry is octant 0's mirrored in the axes where qt
// has a bit set (d -> mirror(d), q -> q ^ qt), so the cell offset, and with it
// the operator T_e, is octant 0's.  m2l_step gives, per step of that order, the
// operator index o (offset + (3,3,3) in base 7), the parent-neighbour slot dn
// (0..26) of the mirrored neighbour and the mirrored source octant qs.
struct M2lSteps {
    int8_t d[189], q[189];
};
constexpr M2lSteps m2l_steps() {
    M2lSteps t{};
    int st = 0;
    for (int d = 0; d < 27; ++d) {
        const int dx = d % 3 - 1, dy = (d / 3) % 3 - 1, dz = d / 9 - 1;
        for (int q = 0; q < 8; ++q) {
            const int ex = 2 * dx - (q & 1), ey = 2 * dy - ((q >> 1) & 1), ez = 2 * dz - ((q >> 2) & 1);
            if (ex >= -1 && ex <= 1 && ey >= -1 && ey <= 1 && ez >= -1 && ez <= 1) continue;  // adjacent: near field
            t.d[st] = static_cast<int8_t>(d);
            t.q[st] = static_cast<int8_t>(q);
            ++st;
        }
    }
    return t;
}
static __constant__ const M2lSteps c_m2l_steps = m2l_steps();
struct M2lStep {
    int o, dn, qs;
};
__host__ __device__ inline M2lStep m2l_step(int d, int q, int qt) {
    const int dx = d % 3 - 1, dy = (d / 3) % 3 - 1, dz = d / 9 - 1;
    const int ex = 2 * dx - (q & 1), ey = 2 * dy - ((q >> 1) & 1), ez = 2 * dz - ((q >> 2) & 1);
    const int mx = (qt & 1) ? -dx : dx, my = (qt & 2) ? -dy : dy, mz = (qt & 4) ? -dz : dz;
    return {(ex + 3) + 7 * (ey + 3) + 49 * (ez + 3), (mx + 1) + 3 * (my + 1) + 9 * (mz + 1), q ^ qt};
}
// The steps of octant qt into o, dn, qs by a block of nth threads.
__device__ inline void m2l_walk(int tid, int nth, int qt, int16_t *o, int16_t *dn, int16_t *qs) {
    for (int st = tid; st < 189; st += nth) {
        const M2lStep s = m2l_step(c_m2l_steps.d[st], c_m2l_steps.q[st], qt);
        o[st] = static_cast<int16_t>(s.o);
        dn[st] = static_cast<int16_t>(s.dn);
        qs[st] = static_cast<int16_t>(s.qs);
    }
}
// The steps st whose live(st) holds, in order, into list, their number into
// *n: called by every thread of a block of at least 192; list, n and the 3 words
// of count in LDS.  Ends with a barrier.
template <class F>
__device__ inline void m2l_live_steps(int tid, int16_t *list, int *n, int *count, F &&live) {
    const bool on = tid < 189 && live(tid);
    const uint64_t b = __ballot(on);
    if (tid < 192 && (tid & 63) == 0) count[tid >> 6] = __popcll(b);
    __syncthreads();
    if (on) list[(tid > 63 ? count[0] : 0) + (tid > 127 ? count[1] : 0) + __popcll(b & ((1ull << (tid & 63)) - 1))] = static_cast<int16_t>(tid);
    if (tid == 0) *n = count[0] + count[1] + count[2];
    __syncthreads();
}

// The mirrored operator is D_qt T_e D_qt with D_qt diagonal +-1; its entry for
// real-packed coefficient k (x -> -x: (-1)^m on cosine, -(-1)^m on sine
// coefficients; y -> -y: -1 on sine; z -> -z: (-1)^(n+m)).
__host__ __device__ inline int m2l_mirror_sign(int qt, int k) {
    int nn = 0;  // k = n^2 + r: degree n, r = 0 (m = 0), 2m - 1 (cosine) or 2m (sine)
    while ((nn + 1) * (nn + 1) <= k) ++nn;
    const int r = k - nn * nn, m = (r + 1) >> 1;
    const bool im = r > 0 && (r & 1) == 0;
    int sg = 1;
    if (qt & 1) sg *= ((m & 1) ? -1 : 1) * (im ? -1 : 1);
    if ((qt & 2) && im) sg = -sg;
    if ((qt & 4) && ((nn + m) & 1)) sg = -sg;
    return sg;
}

}  // namespace vg
