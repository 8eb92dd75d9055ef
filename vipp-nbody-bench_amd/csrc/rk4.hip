// rk4.hip - FP64 classic RK4 on the caller-ordered state, energies and work counts.
//
// The stage arithmetic is the reference's (solver_ref.hpp:36-104):
//   x_out += (dt/6) v ; v_out += (dt/6) a      after the stage-0 force
//   x = x0 + v (dt/2) ; v = v0 + a (dt/2)      (euler, solver_ref.hpp:109-112)
//   ... (dt/3, dt/2), (dt/3, dt), (dt/6, copy out)
// evaluated with the same roundings: contraction into FMA is off here, so the
// FP64 state matches a non-FMA x86 build of the reference bit for bit when the
// forces agree.
#include "gravity.hpp"

#pragma clang fp contract(off)

namespace vg {
namespace {

// accumulate with weight cw, then take the next Euler state with step h (last
// stage: copy the accumulated state out instead).  The first stage keeps the
// state it finds as x0 and v0 and accumulates from it.  Grid-stride over the
// 3n scalars; each block also leaves the partial bounding box of the positions
// it wrote (7 doubles at part, the layout of k_aabb), so the next tree build
// needs no pass of its own over x.
template <class A>
__global__ __launch_bounds__(256) void k_rk4_stage(int64_t n3, double cw, double h, bool first, bool last, const A *__restrict__ a, double *__restrict__ x,
                                                   double *__restrict__ v, double *__restrict__ x0, double *__restrict__ v0,
                                                   double *__restrict__ xo, double *__restrict__ vo, double *__restrict__ part) {
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    double bad = 0;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    const int s3 = static_cast<int>(stride % 3);
    int64_t i = blockIdx.x * 256ll + threadIdx.x;
    int comp = static_cast<int>(i % 3);
    for (; i < n3; i += stride) {
        const double ai = static_cast<double>(a[i]);
        const double vi = v[i], xi = first ? x[i] : 0.0;
        const double xon = (first ? xi : xo[i]) + cw * vi;
        const double von = (first ? vi : vo[i]) + cw * ai;
        double xn;
        if (last) {
            xn = xon;
            v[i] = von;
        } else {
            xo[i] = xon;
            vo[i] = von;
            if (first) {
                x0[i] = xi;
                v0[i] = vi;
            }
            xn = (first ? xi : x0[i]) + vi * h;
            v[i] = (first ? vi : v0[i]) + ai * h;
        }
        x[i] = xn;
        if (!isfinite(xn)) bad = 1;
        lo[0] = comp == 0 ? fmin(lo[0], xn) : lo[0];
        lo[1] = comp == 1 ? fmin(lo[1], xn) : lo[1];
        lo[2] = comp == 2 ? fmin(lo[2], xn) : lo[2];
        hi[0] = comp == 0 ? fmax(hi[0], xn) : hi[0];
        hi[1] = comp == 1 ? fmax(hi[1], xn) : hi[1];
        hi[2] = comp == 2 ? fmax(hi[2], xn) : hi[2];
        comp += s3;
        if (comp >= 3) comp -= 3;
    }
    aabb_block_store(lo, hi, bad, part + 7ll * blockIdx.x);
}

// The largest finite |m| of each block's share, in pinned host memory.
__global__ __launch_bounds__(256) void k_largest_mass(int64_t n, const double *__restrict__ m, double *part) {
    __shared__ double s[256];
    double v = 0;
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll)
        if (isfinite(m[i])) v = fmax(v, fabs(m[i]));
    s[threadIdx.x] = v;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < static_cast<unsigned>(w)) s[threadIdx.x] = fmax(s[threadIdx.x], s[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// FP64 block sums of m |v|^2 (the first half of the grid) and m pot (the second) into
// pinned host memory: one launch and one wait, where two of each, a copy and a device
// allocation took 56 us of the 995 that the energies of 256k particles took.
constexpr int EN_BLOCKS = 256;
__global__ __launch_bounds__(256) void k_energy(int64_t n, const double *__restrict__ v, const double *__restrict__ m, double mass,
                                                const double *__restrict__ pot, double *part) {
    __shared__ double s[256];
    const bool kinetic = blockIdx.x < EN_BLOCKS;
    double acc = 0;
    for (int64_t i = blockIdx.x % EN_BLOCKS * 256ll + threadIdx.x; i < n; i += EN_BLOCKS * 256) {
        const double mi = m ? m[i] : mass;
        if (kinetic)
            acc += mi * (v[3 * i] * v[3 * i] + v[3 * i + 1] * v[3 * i + 1] + v[3 * i + 2] * v[3 * i + 2]);
        else
            acc += mi * pot[i];
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < static_cast<unsigned>(w)) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// work counts: [0] P2P pairs (i != j), [1] M2L pairs of targets at level >= 2,
// [2] M2L pairs whose target and source both hold particles, [3] list
// entries stored (AP, NB and each cell's own NI entries)
__global__ __launch_bounds__(256) void k_count(int64_t nc, const int8_t *__restrict__ level, const int32_t *__restrict__ child, const uint32_t *__restrict__ count,
                                               const int32_t *__restrict__ anc, const int32_t *__restrict__ ni, const int32_t *__restrict__ ni_cnt,
                                               const int32_t *__restrict__ ap, const int32_t *__restrict__ ap_cnt, const int32_t *__restrict__ nb_cnt,
                                               unsigned long long *__restrict__ out) {
    const int64_t c = blockIdx.x * 256ll + threadIdx.x;
    unsigned long long pairs = 0, m2l = 0, live = 0, entries = 0;
    if (c < nc) {
        entries = static_cast<unsigned long long>(ap_cnt[c] + nb_cnt[c] + ni_cnt[c]);
        if (level[c] >= 2) {
            m2l = static_cast<unsigned long long>(ap_cnt[c]);
            if (count[c] > 0)
                for (int e = 0; e < ap_cnt[c]; ++e) live += count[ap[189 * c + e]] > 0;
        }
        if (child[c] < 0 && count[c] > 0) {
            unsigned long long src = 0;
            for (int l = 0; l <= level[c]; ++l) {
                const int32_t a = anc[c * (MAXD + 1) + l];
                for (int e = 0; e < ni_cnt[a]; ++e) src += count[ni[27 * static_cast<int64_t>(a) + e]];
            }
            pairs = static_cast<unsigned long long>(count[c]) * (src - 1);
        }
    }
    if (pairs) atomicAdd(&out[0], pairs);
    if (m2l) atomicAdd(&out[1], m2l);
    if (live) atomicAdd(&out[2], live);
    if (entries) atomicAdd(&out[3], entries);
}

}  // namespace

void rk4_stage(Ctx &c, int stage, double dt) {
    const int64_t n3 = 3 * c.n;
    // weights and Euler steps of solver_ref.hpp:58-99
    const double cw = (stage == 0 || stage == 3) ? dt / 6 : dt / 3;
    const double h = stage == 2 ? dt : dt / 2;
    const bool first = stage == 0, last = stage == 3;
    const int nb = static_cast<int>(std::min<int64_t>(1024, std::max<int64_t>(1, ceil_div(n3, 256))));
    c.aabb_part.ensure(7 * static_cast<size_t>(nb));
    c.aabb_parts = 0;
    if (c.prec == 0)
        k_rk4_stage<double><<<nb, 256, 0, c.stream>>>(n3, cw, h, first, last, c.acc64, c.x, c.v, c.x0, c.v0, c.xo, c.vo, c.aabb_part);
    else
        k_rk4_stage<float><<<nb, 256, 0, c.stream>>>(n3, cw, h, first, last, c.acc32, c.x, c.v, c.x0, c.v0, c.xo, c.vo, c.aabb_part);
    VG_LAUNCH_CHECK();
    c.aabb_parts = nb;
}

double largest_mass(Ctx &c) {
    double *part = reinterpret_cast<double *>(static_cast<char *>(c.pinned) + Ctx::PINNED_ENERGY);
    k_largest_mass<<<EN_BLOCKS, 256, 0, c.stream>>>(c.n, c.m, part);
    VG_LAUNCH_CHECK();
    VG_HIP(hipStreamSynchronize(c.stream));
    return *std::max_element(part, part + EN_BLOCKS);
}

void energies(Ctx &c, double &kinetic, double &potential) {
    double *part = reinterpret_cast<double *>(static_cast<char *>(c.pinned) + Ctx::PINNED_ENERGY);
    static_assert(Ctx::PINNED_ENERGY + 2 * EN_BLOCKS * sizeof(double) <= Ctx::PINNED_BYTES - 64, "pinned words");
    k_energy<<<2 * EN_BLOCKS, 256, 0, c.stream>>>(c.n, c.v, c.has_masses ? c.m.p : nullptr, c.mass, c.pot64.p, part);
    VG_LAUNCH_CHECK();
    VG_HIP(hipStreamSynchronize(c.stream));
    double ke = 0, pe = 0;
    for (int b = 0; b < EN_BLOCKS; ++b) ke += part[b];  // fixed order: deterministic
    for (int b = 0; b < EN_BLOCKS; ++b) pe += part[EN_BLOCKS + b];
    kinetic = 0.5 * ke;
    potential = -0.5 * c.G * pe;
}

void count_work(Ctx &c) {
    TreeDev &t = c.t;
    DevBuf<unsigned long long> out;
    out.ensure(4);
    VG_HIP(hipMemsetAsync(out.p, 0, 4 * sizeof(unsigned long long), c.stream));
    k_count<<<ceil_div(t.ncells, 256), 256, 0, c.stream>>>(t.ncells, t.level, t.child, t.count, t.anc, t.ni, t.ni_cnt, t.ap, t.ap_cnt, t.nb_cnt, out);
    VG_LAUNCH_CHECK();
    unsigned long long h[4];
    VG_HIP(hipMemcpyAsync(h, out.p, sizeof(h), hipMemcpyDeviceToHost, c.stream));
    VG_HIP(hipStreamSynchronize(c.stream));
    c.counts[0] = static_cast<double>(h[0]);
    c.counts[1] = static_cast<double>(h[1]);
    c.counts[2] = static_cast<double>(t.ncells);
    c.counts[3] = static_cast<double>(t.nleaves);
    c.counts[4] = static_cast<double>(t.depth);
    c.counts[5] = static_cast<double>(h[2]);
    c.counts[7] = static_cast<double>(h[3]);
}

}  // namespace vg
