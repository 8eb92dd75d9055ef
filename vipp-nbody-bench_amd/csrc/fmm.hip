// fmm.hip - expansions and translations of the gravity FMM.
//
// Conventions follow the reference (fmm.hpp:167-374): Y_n^m is
// sqrt((n-|m|)!/(n+|m|)!) P_n^{|m|}(cos a) e^{i m b} with the Condon-Shortley
// phase, A_n^m = (-1)^n / sqrt((n-|m|)!(n+|m|)!), and
//   P2M  M_n^m = sum_i m_i rho_i^n Y_n^{-m}                       (fmm.hpp:224-244)
//   M2M  Greengard's shift with i^{|k|-|m|-|k-m|}                  (fmm.hpp:247-274)
//   M2L  L_j^k = sum M_n^m i^{|k-m|-|k|-|m|} A_n^m A_j^k Y_{j+n}^{m-k}
//              / ((-1)^n A_{j+n}^{m-k} rho^{j+n+1})                (fmm.hpp:277-304)
//   L2L  with i^{|m|-|m-k|-|k|}                                   (fmm.hpp:307-329)
//   L2P  gradient of sum L_l^m r^l Y_l^m                           (fmm.hpp:332-374)
// Storage differs: only m >= 0 is kept (M_n^{-m} = conj M_n^m), as (p+1)^2
// reals per cell, and every expansion is scaled by the cell width w of its
// level (M~_n = M_n / w^n, L~_j = L_j w^{j+1}).  Then every operator depends
// only on the cell offset in units of w, which is the same at every level
// (all levels share the root box's aspect ratio), so one set of operators
// (8 M2M, 8 L2L, 316 M2L) serves the whole tree.  Operators are built in FP64
// on the device for the current root box before each evaluation.
// Solid harmonics R_n^m = r^n Y_n^m are evaluated with Cartesian recurrences
// (no trigonometry), gradients with the ladder relations
//   dR_n^m/dz = sqrt((n+m)(n-m)) R_{n-1}^m,
//   (d/dx + i d/dy) R_n^m = sqrt((n-m)(n-m-1)) R_{n-1}^{m+1},
//   (d/dx - i d/dy) R_n^m = -sqrt((n+m)(n+m-1)) R_{n-1}^{m-1}   (m >= 1).
#include "gravity.hpp"

#include <cmath>
#include <mutex>

namespace vg {
namespace {

constexpr int AL = 2 * MAXP;        // A_n^m needed up to n = 2p
constexpr int AW = 2 * AL + 1;
__constant__ double cA[(AL + 1) * AW];
// R recurrences of P2M: diag[m], r1[n][m], r2[n][m]
__constant__ double cDiag[MAXP + 1], cR1[(MAXP + 1) * (MAXP + 1)], cR2[(MAXP + 1) * (MAXP + 1)];

struct dc {
    double re, im;
};
__device__ inline dc cmul(dc a, dc b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ inline dc cconj(dc a) { return {a.re, -a.im}; }
__device__ inline dc cscale(dc a, double s) { return {a.re * s, a.im * s}; }
__device__ inline dc cadd(dc a, dc b) { return {a.re + b.re, a.im + b.im}; }
__device__ inline dc csub(dc a, dc b) { return {a.re - b.re, a.im - b.im}; }

__device__ inline double Acoef(int n, int m) { return cA[n * AW + AL + m]; }
__device__ inline double ipow_even(int e) { return ((e / 2) % 2 == 0) ? 1.0 : -1.0; }

// Y_l^mu of the reference (fmm.hpp:169-194) for one direction; tab holds m >= 0
// at l(l+1)/2 + m as (re, im).
__device__ inline dc Yget(const double *tab, int l, int mu) {
    const int am = mu < 0 ? -mu : mu;
    const dc v{tab[2 * (l * (l + 1) / 2 + am)], tab[2 * (l * (l + 1) / 2 + am) + 1]};
    return mu < 0 ? cconj(v) : v;
}

constexpr int HSTRIDE = 2 * ((AL + 1) * (AL + 2) / 2) + 2;  // per offset: Y table + rho

// Y_l^m(direction) for l <= lmax and |v| of each offset vector.
// One thread per (offset, m): P_l^m by the upward recurrence in l, with
// P_m^m = (-1)^m (2m-1)!! sin^m, and sqrt((l-m)!/(l+m)!) carried along l.
// Offset vectors in units of a level's x width, the cell aspect ratio being
// (1, ry, rz): 0..7 M2M (child centre - parent centre of child octant o),
// 8..15 L2L (their negatives), 16 + o M2L (source - target cell, o in base 7
// holding (dx + 3, dy + 3, dz + 3)).
__global__ __launch_bounds__(64) void k_harmonics(const int16_t *__restrict__ sel, int nvec, const double *__restrict__ box, int lmax, double *__restrict__ out) {
    const int o = sel[blockIdx.x];  // the vectors any kernel reads (see operators_build)
    const int m = threadIdx.x;
    if (o >= nvec || m > lmax) return;
    const double wx = box[3] - box[0], wy = box[4] - box[1], wz = box[5] - box[2];
    const double ry = wx > 0 ? wy / wx : 1.0, rz = wx > 0 ? wz / wx : 1.0;
    double vx, vy, vz;
    if (o < 16) {
        const int q = o & 7;
        const double cx = (q & 1) ? -0.25 : 0.25, cy = ((q >> 1) & 1) ? -0.25 * ry : 0.25 * ry, cz = ((q >> 2) & 1) ? -0.25 * rz : 0.25 * rz;
        vx = o < 8 ? cx : -cx;
        vy = o < 8 ? cy : -cy;
        vz = o < 8 ? cz : -cz;
    } else {
        const int e = o - 16;
        vx = e % 7 - 3;
        vy = ((e / 7) % 7 - 3) * ry;
        vz = (e / 49 - 3) * rz;
    }
    double *tab = out + static_cast<size_t>(o) * HSTRIDE;
    const double rho = sqrt(vx * vx + vy * vy + vz * vz);
    if (m == 0) {
        tab[HSTRIDE - 2] = rho;
        tab[HSTRIDE - 1] = 0;
    }
    const double rxy = sqrt(vx * vx + vy * vy);
    const double ct = rho > 0 ? vz / rho : 1.0, st = rho > 0 ? rxy / rho : 0.0;
    const dc eph = rxy > 0 ? dc{vx / rxy, vy / rxy} : dc{1.0, 0.0};
    dc em{1.0, 0.0};  // e^{i m phi}
    double pmm = 1.0, f = 1.0;  // P_m^m, (l-m)!/(l+m)! at l = m: 1/(2m)!
    for (int i = 1; i <= m; ++i) {
        pmm *= -(2.0 * i - 1) * st;
        em = cmul(em, eph);
        f /= (2.0 * i - 1) * (2.0 * i);
    }
    double p0 = 0, p1 = pmm;
    for (int l = m; l <= lmax; ++l) {
        double pl;
        if (l == m)
            pl = pmm;
        else if (l == m + 1)
            pl = ct * (2.0 * m + 1) * pmm;
        else
            pl = ((2.0 * l - 1) * ct * p1 - (l + m - 1.0) * p0) / (l - m);
        if (l > m) {
            p0 = p1;
            p1 = pl;
            f *= static_cast<double>(l - m) / static_cast<double>(l + m);
        }
        const double nrm = sqrt(f) * pl;
        tab[2 * (l * (l + 1) / 2 + m)] = nrm * em.re;
        tab[2 * (l * (l + 1) / 2 + m) + 1] = nrm * em.im;
    }
}

// Row r of an operator in the real-packed basis: degree j, order k, part
// 0 = Re (cosine) or 1 = Im (sine).  Column pair (n, m): Re at kidx_re, Im at
// kidx_im, from the complex coefficients T(+m), T(-m).
__device__ inline void row_of(int r, int &j, int &k, int &part) {
    j = static_cast<int>(sqrt(static_cast<double>(r)));
    while (j * j > r) --j;
    while ((j + 1) * (j + 1) <= r) ++j;
    const int q = r - j * j;
    if (q == 0) {
        k = 0;
        part = 0;
    } else {
        k = (q + 1) / 2;
        part = (q % 2 == 1) ? 0 : 1;
    }
}

// FP32 M2L operators are kept in the order in which k_m2l_f32's lanes read
// them: per operator RT x NJ fragments (16 rows, 16 columns) of 64 lanes x 4
// columns.  Lane 16 q + row holds columns 4 q .. 4 q + 3 of the fragment, so
// that its four words are the operands of four products v_mfma_f32_16x16x4;
// the last column group has only the nks = ceil(rest / 4) products it needs,
// lane 16 q + row then holds columns nks q .. nks q + nks - 1.
struct OpFrag {
    int nt, nks;  // 16-row tiles (and 16-column groups), products of the last group
    __host__ __device__ explicit OpFrag(int K) : nt((K + 15) / 16), nks((K - 16 * ((K + 15) / 16 - 1) + 3) / 4) {}
    __host__ __device__ size_t size() const { return static_cast<size_t>(nt) * nt * 256; }
    __host__ __device__ size_t at(int r, int c) const {
        const int j = c >> 4, w = j + 1 < nt ? 4 : nks;
        return (static_cast<size_t>((r >> 4) * nt + j) * 64 + (c & 15) / w * 16 + (r & 15)) * 4 + (c & 15) % w;
    }
};

// FP32 M2M and L2L operators, in the order in which k_ml_f32's lanes read them: fragments
// as above, but lane 16 q + row holds the columns 4 i + q, i = 0 .. 3, so that the
// products go through the columns in order.
struct MlFrag {
    int nt;
    __host__ __device__ explicit MlFrag(int K) : nt((K + 15) / 16) {}
    __host__ __device__ size_t size() const { return static_cast<size_t>(nt) * nt * 256; }
    __host__ __device__ size_t at(int r, int c) const { return (static_cast<size_t>((r >> 4) * nt + (c >> 4)) * 64 + (c & 3) * 16 + (r & 15)) * 4 + (c & 15) / 4; }
};

// op block layout: [M2M 0..7][L2L 8..15][M2L 16..16+342], each K*K; M2L
// blocks row-major [row][col], M2M and L2L blocks column-major [col][row] (their
// kernels give each lane one output row, so lanes then read consecutive words).
// With frag (FP32): M2M and L2L blocks in op in MlFrag's order, M2L blocks in frag
// in OpFrag's; what no column pair fills stays as it is there, zero.
// One block per (operator, OPS_ROWS rows), 128 threads per row r; thread t of
// a row takes the column pair (n, m >= 0) number t, i.e. the real-packed
// columns of degree n, order m.
constexpr int OPS_ROWS = 4;
template <class R>
__global__ __launch_bounds__(128 * OPS_ROWS) void k_ops(const int16_t *__restrict__ sel, const double *__restrict__ harm, int p, int K, R *__restrict__ op,
                                                         R *__restrict__ frag) {
    const int blk = sel[blockIdx.x];  // operator index
    const int r = blockIdx.y * OPS_ROWS + static_cast<int>(threadIdx.x >> 7);
    const int t = threadIdx.x & 127;
    const bool cmaj = blk < 16;
    const OpFrag fr(K);
    const MlFrag ml(K);
    const bool fragment = frag != nullptr;
    R *dst = cmaj ? op + static_cast<size_t>(blk) * K * K + r : op + (static_cast<size_t>(blk) * K + r) * K;
    const size_t cs = cmaj ? static_cast<size_t>(K) : 1;  // column stride
    if (r < K && !fragment)
        for (int c = t; c < K; c += 128) dst[c * cs] = R(0);
    __syncthreads();
    if (r >= K) return;
    int j, k, part;
    row_of(r, j, k, part);
    if (t >= (p + 1) * (p + 2) / 2) return;
    int n = 0;
    while ((n + 1) * (n + 2) / 2 <= t) ++n;
    const int mp = t - n * (n + 1) / 2;  // column pair (n, mp)
    const double *tab = harm + static_cast<size_t>(blk) * HSTRIDE;
    const double rho = tab[HSTRIDE - 2];
    dc tpm[2] = {{0, 0}, {0, 0}};
    if (blk < 8) {
        // M2M, child offset q: column (j', k') = (n, mp) of the child expansion, scaled by 2^{-j'} (fmm.hpp:256-270)
        const int jp = n, kp = mp;
        if (jp > j) return;
        const int nn = j - jp;
        const double rn = pow(rho, nn);
        const double scale = ldexp(1.0, -jp);
        for (int sgn = 0; sgn < 2; ++sgn) {
            const int kk = sgn == 0 ? kp : -kp;
            const int m = k - kk;
            if (m < -nn || m > nn) continue;
            const double coef = ipow_even(abs(k) - abs(m) - abs(k - m)) * Acoef(nn, m) * Acoef(jp, kk) * rn / Acoef(j, k) * scale;
            tpm[sgn] = cscale(Yget(tab, nn, -m), coef);
        }
    } else if (blk < 16) {
        // L2L, child offset q: column (n, m) of the parent expansion, scaled by 2^{-(j+1)} (fmm.hpp:313-327)
        if (n < j) return;
        const double scale = ldexp(1.0, -(j + 1));
        const double rn = pow(rho, n - j);
        for (int sgn = 0; sgn < 2; ++sgn) {
            const int m = sgn == 0 ? mp : -mp;
            if (m - k < -(n - j) || m - k > n - j) continue;
            const double coef = ipow_even(abs(m) - abs(m - k) - abs(k)) * Acoef(n - j, m - k) * Acoef(j, k) * rn /
                                (((n + j) % 2 ? -1.0 : 1.0) * Acoef(n, m)) * scale;
            tpm[sgn] = cscale(Yget(tab, n - j, m - k), coef);
        }
    } else {
        // M2L, offset o (fmm.hpp:287-302); rows of the 27 near offsets stay zero
        const int o = blk - 16;
        const int ox = o % 7 - 3, oy = (o / 7) % 7 - 3, oz = o / 49 - 3;
        if (ox >= -1 && ox <= 1 && oy >= -1 && oy <= 1 && oz >= -1 && oz <= 1) return;
        const double rj = pow(rho, j + n + 1);
        for (int sgn = 0; sgn < 2; ++sgn) {
            if (mp == 0 && sgn == 1) continue;
            const int m = sgn == 0 ? mp : -mp;
            const double coef = ipow_even(abs(k - m) - abs(k) - abs(m)) * Acoef(n, m) * Acoef(j, k) / ((n % 2 ? -1.0 : 1.0) * Acoef(j + n, m - k) * rj);
            tpm[sgn] = cscale(Yget(tab, j + n, m - k), coef);
        }
    }
    // the pair's real-packed columns (each written by this thread only)
    auto put = [&](int c, double v) {
        if (fragment && cmaj)
            op[blk * ml.size() + ml.at(r, c)] = static_cast<R>(v);
        else if (fragment)
            frag[(blk - 16) * fr.size() + fr.at(r, c)] = static_cast<R>(v);
        else
            dst[c * cs] = static_cast<R>(v);
    };
    if (mp == 0) {
        put(kidx_re(n, 0), part == 0 ? tpm[0].re : tpm[0].im);
    } else {
        const dc sum = cadd(tpm[0], tpm[1]), dif = csub(tpm[0], tpm[1]);
        put(kidx_re(n, mp), part == 0 ? sum.re : sum.im);
        put(kidx_im(n, mp), part == 0 ? -dif.im : dif.re);
    }
}

// ---------------------------------------------------------------------------
// P2M: one wavefront per leaf.  Lane = g NM + i, i < NM = p / 2 + 1: particle
// group g (G = 64 / NM groups, particles g, g + G, ...) and the order pair
// (m1, m2) = (i, p - i), so that every lane walks the same number of
// recurrence steps: R_{m1}^{m1} .. R_p^{m1} (p - m1 + 1 values), then
// R_{m2}^{m2} .. R_p^{m2} (p - m2 + 1; none when m2 = m1), p + 2 in all.
// Every lane forms the diagonal R_q^q, q <= p, and keeps the two it starts
// from; step s accumulates m_i conj(R) into accumulator s.  The groups are
// then summed in fixed order through LDS by all 64 lanes.
// ---------------------------------------------------------------------------
template <class R, int P>
__global__ __launch_bounds__(256) void k_p2m(const int32_t *__restrict__ leaves, int nleaves, const int8_t *__restrict__ level,
                                             const uint32_t *__restrict__ start, const uint32_t *__restrict__ count, const double *__restrict__ bmin,
                                             const double *__restrict__ bmax, const double *__restrict__ xs64, double wx0, int K, int ldk,
                                             R *__restrict__ M, uint16_t *__restrict__ Ms) {
    constexpr int p = P;       // the order is a template argument, so the recurrence unrolls fully
    constexpr int NS = P + 2;  // recurrence steps per lane
    __shared__ R red[4][64][2 * NS];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int li = blockIdx.x * 4 + w;
    if (li >= nleaves) return;  // whole wavefront: no barrier below spans wavefronts
    const int32_t c = leaves[li];
    if (level[c] < 2) return;  // solver_ref.hpp:187-188
    const int NM = p / 2 + 1, G = 64 / NM;
    const int i = lane % NM, g = lane / NM;
    const bool act = g < G;
    const int m1 = i, m2 = p - i;
    const int len1 = p - m1 + 1, len2 = m2 != m1 ? p - m2 + 1 : 0, tot = len1 + len2;
    const uint32_t s = start[c], cnt = count[c];
    const double iw = 1.0 / ldexp(wx0, -level[c]);
    const double cx = (bmin[3 * c] + bmax[3 * c]) / 2, cy = (bmin[3 * c + 1] + bmax[3 * c + 1]) / 2, cz = (bmin[3 * c + 2] + bmax[3 * c + 2]) / 2;
    // R_m^m = (prod_{q<=m} cDiag[q]) (x + i y)^m: the products for m1 and m2
    double sc1 = 1.0, sc2 = 1.0;
    for (int q = 1; q <= m2; ++q) {
        if (q <= m1) sc1 *= cDiag[q];
        sc2 *= cDiag[q];
    }
    const R s1 = static_cast<R>(sc1), s2 = static_cast<R>(sc2);
    // recurrence coefficients of each step (unused at the two chain starts)
    R c1[NS], c2[NS], are[NS], aim[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int n = k < len1 ? m1 + k : m2 + (k - len1), m = k < len1 ? m1 : m2;
        const int idx = (k < tot && n <= MAXP) ? n * (MAXP + 1) + m : 0;
        c1[k] = static_cast<R>(cR1[idx]);
        c2[k] = static_cast<R>(cR2[idx]);
        are[k] = 0;
        aim[k] = 0;
    }
    if (act) {
        // the next particle of this lane group is loaded before the current
        // one's harmonics are formed, so its latency hides behind them
        const double2 *xs2 = reinterpret_cast<const double2 *>(xs64);
        double2 nxy = make_double2(0, 0), nzm = make_double2(0, 0);
        if (g < cnt) {
            nxy = xs2[2 * static_cast<size_t>(s + g)];
            nzm = xs2[2 * static_cast<size_t>(s + g) + 1];
        }
        for (uint32_t j = g; j < cnt; j += G) {
            const double2 cxy = nxy, czm = nzm;
            if (j + G < cnt) {
                nxy = xs2[2 * static_cast<size_t>(s + j + G)];
                nzm = xs2[2 * static_cast<size_t>(s + j + G) + 1];
            }
            const R x = static_cast<R>((cxy.x - cx) * iw), y = static_cast<R>((cxy.y - cy) * iw), z = static_cast<R>((czm.x - cz) * iw);
            const R mi = static_cast<R>(czm.y);
            const R r2 = x * x + y * y + z * z;
            // (x + i y)^m1 and ^m2 by repeated squaring: w^(2^b) once, a
            // multiply per set bit of each exponent (selects, no branches)
            R d1re = 1, d1im = 0, d2re = 1, d2im = 0;
            {
                R wre = x, wim = y;  // w^(2^b)
                for (int b = 0; (1 << b) <= p; ++b) {
                    const R t1re = d1re * wre - d1im * wim, t1im = d1re * wim + d1im * wre;
                    const R t2re = d2re * wre - d2im * wim, t2im = d2re * wim + d2im * wre;
                    const bool u1 = (m1 >> b) & 1, u2 = (m2 >> b) & 1;
                    d1re = u1 ? t1re : d1re;
                    d1im = u1 ? t1im : d1im;
                    d2re = u2 ? t2re : d2re;
                    d2im = u2 ? t2im : d2im;
                    const R sre = wre * wre - wim * wim, sim = 2 * wre * wim;
                    wre = sre;
                    wim = sim;
                }
            }
            d1re *= s1;
            d1im *= s1;
            d2re *= s2;
            d2im *= s2;
            R bre = 0, bim = 0, cre = 0, cim = 0;  // R_{n-2}^m, R_{n-1}^m
#pragma unroll
            for (int st = 0; st < NS; ++st) {
                if (st > p + 1) break;
                if (st == 0) {
                    cre = d1re;
                    cim = d1im;
                } else {
                    // the second chain starts at step len1: R_{m2}^{m2}, with R_{m2-1}^{m2} = 0
                    const bool rs = st == len1;
                    const R nre = c1[st] * z * cre - c2[st] * r2 * bre, nim = c1[st] * z * cim - c2[st] * r2 * bim;
                    bre = rs ? R(0) : cre;
                    bim = rs ? R(0) : cim;
                    cre = rs ? d2re : nre;
                    cim = rs ? d2im : nim;
                }
                if (st < tot) {
                    are[st] += mi * cre;
                    aim[st] -= mi * cim;  // conj
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        red[w][lane][2 * k] = are[k];
        red[w][lane][2 * k + 1] = aim[k];
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // output (i, step, part) summed over the groups in fixed order
    R *out = M + static_cast<size_t>(c) * ldk;
    for (int o = lane; o < NM * NS * 2; o += 64) {
        const int oi = o / (2 * NS), ost = (o / 2) % NS, part = o & 1;
        const int om1 = oi, om2 = p - oi, ol1 = p - om1 + 1, ol2 = om2 != om1 ? p - om2 + 1 : 0;
        if (ost >= ol1 + ol2) continue;
        const int n = ost < ol1 ? om1 + ost : om2 + (ost - ol1), m = ost < ol1 ? om1 : om2;
        if (part == 1 && m == 0) continue;
        R sum = 0;
        for (int gg = 0; gg < G; ++gg) sum += red[w][gg * NM + oi][2 * ost + part];
        const int at = part == 0 ? kidx_re(n, m) : kidx_im(n, m);
        out[at] = sum;
        if (Ms) {  // split mode: M2L's halves too
            uint32_t h, l;
            split_m(static_cast<float>(sum), h, l);
            Ms[static_cast<size_t>(c) * 2 * ldk + at] = static_cast<uint16_t>(h);
            Ms[static_cast<size_t>(c) * 2 * ldk + ldk + at] = static_cast<uint16_t>(l);
        }
    }
    for (int q = K + lane; q < ldk; q += 64) {
        out[q] = R(0);
        if (Ms) Ms[static_cast<size_t>(c) * 2 * ldk + q] = Ms[static_cast<size_t>(c) * 2 * ldk + ldk + q] = 0;
    }
}

// FP64 M2M (solver_ref.hpp:196-197) and L2L of the internal cells of one tree level, PB parents per block: every operator word read
// from L2 serves PB parents, and PB is chosen per level (pick_pb) so that the
// launch still has enough blocks to fill the chip.  Operator blocks are
// column-major, so the lanes (output rows) read consecutive words; the
// staged expansions are [col][parent] so a lane reads its PB inputs as vectors.
template <int PB>
__global__ __launch_bounds__(256) void k_m2m(const int32_t *__restrict__ ids, int nids, const int32_t *__restrict__ child,
                                             const uint32_t *__restrict__ count, const double *__restrict__ op, int K, int ldk, double *__restrict__ M) {
    __shared__ double cm[8 * MAXK][PB];  // [child q][col][parent]
    const int p0 = blockIdx.x * PB;
    const int np = min(PB, nids - p0);
    for (int i = threadIdx.x; i < PB * 8 * K; i += 256) {
        const int u = i % PB, qc = i / PB;  // qc = q K + col
        const int q = qc / K, col = qc % K;
        double v = 0;
        if (u < np) {
            const int32_t cb = child[ids[p0 + u]] + q;
            if (count[cb]) v = M[static_cast<size_t>(cb) * ldk + col];
        }
        cm[qc][u] = v;
    }
    __syncthreads();
    for (int r = threadIdx.x; r < K; r += 256) {
        int j = 0;
        while ((j + 1) * (j + 1) <= r) ++j;
        const int cend = (j + 1) * (j + 1);  // output degree j uses child degrees <= j
        double acc[PB];
#pragma unroll
        for (int u = 0; u < PB; ++u) acc[u] = 0;
        for (int q = 0; q < 8; ++q) {
            const double *ocol = op + static_cast<size_t>(q) * K * K + r;
            for (int col = 0; col < cend; ++col) {
                const double a = ocol[static_cast<size_t>(col) * K];
#pragma unroll
                for (int u = 0; u < PB; ++u) acc[u] += a * cm[q * K + col][u];  // empty children are zero
            }
        }
#pragma unroll
        for (int u = 0; u < PB; ++u)
            if (u < np) M[static_cast<size_t>(ids[p0 + u]) * ldk + r] = acc[u];
    }
    for (int i = K + threadIdx.x; i < ldk; i += 256)
        for (int u = 0; u < np; ++u) M[static_cast<size_t>(ids[p0 + u]) * ldk + i] = 0.0;
}

template <int PB>
__global__ __launch_bounds__(256) void k_l2l(const int32_t *__restrict__ ids, int nids, const int32_t *__restrict__ child,
                                             const uint32_t *__restrict__ count, const double *__restrict__ op, int K, int ldk, double *__restrict__ L) {
    __shared__ double pl[MAXK][PB];  // [col][parent]
    const int p0 = blockIdx.x * PB;
    const int np = min(PB, nids - p0);
    for (int i = threadIdx.x; i < PB * K; i += 256) {
        const int u = i % PB, col = i / PB;
        pl[col][u] = u < np ? L[static_cast<size_t>(ids[p0 + u]) * ldk + col] : 0.0;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 8 * K; i += 256) {
        const int q = i / K, r = i % K;
        const double *ocol = op + static_cast<size_t>(8 + q) * K * K + r;
        int j = 0;
        while ((j + 1) * (j + 1) <= r) ++j;
        double acc[PB];
#pragma unroll
        for (int u = 0; u < PB; ++u) acc[u] = 0;
        for (int col = j * j; col < K; ++col) {  // parent degrees >= j
            const double a = ocol[static_cast<size_t>(col) * K];
#pragma unroll
            for (int u = 0; u < PB; ++u) acc[u] += a * pl[col][u];
        }
#pragma unroll
        for (int u = 0; u < PB; ++u) {
            if (u >= np) continue;
            const int32_t cc = child[ids[p0 + u]] + q;
            if (count[cc]) L[static_cast<size_t>(cc) * ldk + r] += acc[u];
        }
    }
}



// ---------------------------------------------------------------------------
// FP64 M2L: targets are the children of octant qt of a chunk of TB internal
// parents; for each well-separated (parent neighbour, source octant) pair the
// (static) cell offset selects one operator, applied as a K x K by K x TB
// product with the gathered source multipoles (offset-grouped GEMM on VALU).
// As on the matrix cores, every block walks octant 0's 189 offsets (m2l_step)
// and the mirror signs D_qt go on the gathered multipoles and on the result,
// so all blocks share 189 operators.  Blocks are placed XCD-aware: the eight
// octant blocks of a parent chunk run side by side on one XCD and share its
// L2.  The prologue tabulates, per parent neighbour and target, the first
// child and the mask of non-empty children, and from them the offsets that
// hold any source; only those are walked.  With nsplit > 1 the walked offsets
// are cut into nsplit consecutive parts, one block each, which write partial
// sums per target slot (parent index * 8 + octant) to part; k_m2l_sum adds
// them in part order.  A thread owns the rows tr + 32 i, i < RPT, and CPT
// consecutive targets; the operator streams through LDS in chunks of KC
// columns, double-buffered through registers (one barrier per chunk), and the
// next offset's first chunk is fetched during the last.
// ---------------------------------------------------------------------------
template <int TB, int RPT>
__global__ __launch_bounds__(256) void k_m2l_plain(const int32_t *__restrict__ parents, int nparents, const int32_t *__restrict__ child,
                                                   const uint32_t *__restrict__ count, const int32_t *__restrict__ nbr27, const double *__restrict__ Mx,
                                                   double *__restrict__ Lx, const double *__restrict__ op, int K, int ldk, int nsplit,
                                                   double *__restrict__ part) {
    using R = double;
    constexpr int KC = 8;                            // operator columns per chunk
    constexpr int CPT = TB / 8;                      // targets per thread
    constexpr int VW = 16 / sizeof(R);               // elements per 16-byte LDS read
    constexpr int SMS = TB + VW;                     // multipole column stride (16-byte rows)
    constexpr int SOS = 32 * RPT + 1;                // operator column stride (odd: no bank conflicts)
    constexpr int NTH = 256;                         // threads
    constexpr int NPF = KC * 32 * RPT / NTH;         // prefetched operator words per thread
    static_assert(CPT % VW == 0 && (KC * 32 * RPT) % NTH == 0, "tile shape");
    extern __shared__ __align__(16) unsigned char m2l_smem[];
    R *sM = reinterpret_cast<R *>(m2l_smem);         // K x SMS: column k of the gathered, signed multipoles
    R *sOp = sM + K * SMS;                           // 2 x KC x SOS: operator columns, transposed
    __shared__ R sg[32 * RPT];                       // D_qt
    __shared__ int32_t s_nc[27 * TB];                // first child of parent neighbour d of target t, or -1
    __shared__ uint8_t s_nm[27 * TB];                // its non-empty children
    __shared__ int32_t tgt[TB];
    __shared__ int16_t s_o[189], s_dn[189], s_qs[189], s_live[189];
    __shared__ int s_nlive, s_cnt[3];
    const int nchunks = (nparents + TB - 1) / TB;
    const int per = nchunks * nsplit;                          // work items per XCD
    const int wi = (blockIdx.x & 7) * per + (blockIdx.x >> 3);  // XCD x takes work items [x W / 8, (x + 1) W / 8)
    if (wi >= 8 * per) return;
    const int sp = wi % nsplit, w = wi / nsplit;  // the parts of one (chunk, octant) are neighbours
    const int chunk = w >> 3, qt = w & 7;
    const int tid = threadIdx.x, tr = tid & 31, tc = tid >> 5;
    m2l_walk(tid, 256, qt, s_o, s_dn, s_qs);
    for (int k = tid; k < 32 * RPT; k += NTH) sg[k] = static_cast<R>(k < K ? m2l_mirror_sign(qt, k) : 0);
    if (tid < TB) {
        const int pi = chunk * TB + tid;
        const int32_t P = pi < nparents ? parents[pi] : -1;
        int32_t t = P >= 0 ? child[P] + qt : -1;
        if (t >= 0 && count[t] == 0) t = -1;
        tgt[tid] = t;
    }
    __syncthreads();
    for (int i = tid; i < 27 * TB; i += NTH) {
        const int d = i / TB, t = i % TB;
        const int pi = chunk * TB + t;
        int32_t cb = -1;
        uint32_t msk = 0;
        if (tgt[t] >= 0) {
            const int32_t sp = nbr27[27 * static_cast<int64_t>(parents[pi]) + d];
            cb = sp >= 0 ? child[sp] : -1;
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
    const int nlive = s_nlive;
    const int lo = sp * nlive / nsplit, hi = (sp + 1) * nlive / nsplit;  // this block's walked offsets
    R acc[RPT][CPT];
#pragma unroll
    for (int i = 0; i < RPT; ++i)
#pragma unroll
        for (int jj = 0; jj < CPT; ++jj) acc[i][jj] = 0;
    const int nkc = (K + KC - 1) / KC;
    const size_t KK = static_cast<size_t>(K) * K;
    R pf[NPF];
    // operator chunk (offset step li, columns [c0, c0 + KC)) into registers:
    // word u of thread tid is row r = i / KC, column c0 + i % KC, i = tid + NTH u
    auto load_op = [&](int li, int c0) {
        const R *O = op + (16 + s_o[s_live[li]]) * KK;
#pragma unroll
        for (int u = 0; u < NPF; ++u) {
            const int i = tid + NTH * u, r = i / KC, c = c0 + i % KC;
            pf[u] = (r < K && c < K) ? O[static_cast<size_t>(r) * K + c] : R(0);
        }
    };
    auto store_op = [&](int b) {
        R *S = sOp + b * KC * SOS;
#pragma unroll
        for (int u = 0; u < NPF; ++u) {
            const int i = tid + NTH * u;
            S[(i % KC) * SOS + i / KC] = pf[u];
        }
    };
    auto fma_col = [&](const R *S, int col) {
        R mv[CPT];
#pragma unroll
        for (int v = 0; v < CPT / VW; ++v) {
            typedef R vec __attribute__((ext_vector_type(VW)));
            const vec x = *reinterpret_cast<const vec *>(sM + col * SMS + tc * CPT + v * VW);
#pragma unroll
            for (int e = 0; e < VW; ++e) mv[v * VW + e] = x[e];
        }
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const R ov = S[tr + 32 * i];
#pragma unroll
            for (int jj = 0; jj < CPT; ++jj) acc[i][jj] += ov * mv[jj];
        }
    };
    if (hi > lo) load_op(lo, 0);
    const int wv = tid >> 6, lane = tid & 63;
    for (int li = lo; li < hi; ++li) {
        const int st = s_live[li], dn = s_dn[st], qs = s_qs[st];
        // gather: wave wv takes targets wv, wv + 4, ..., lanes the columns
        for (int t = wv; t < TB; t += 4) {
            const int32_t cb = s_nc[dn * TB + t];
            const bool has = (s_nm[dn * TB + t] >> qs) & 1;
            const R *src = Mx + static_cast<size_t>(has ? cb + qs : 0) * ldk;
            for (int col = lane; col < K; col += 64) sM[col * SMS + t] = has ? sg[col] * src[col] : R(0);
        }
        store_op(0);
        if (nkc > 1) load_op(li, KC);
        else if (li + 1 < hi) load_op(li + 1, 0);
        __syncthreads();  // multipoles and chunk 0 are in LDS
        for (int kc = 0; kc < nkc; ++kc) {
            const int c0 = kc * KC, b = kc & 1;
            const R *S = sOp + b * KC * SOS;
            if (c0 + KC <= K) {
#pragma unroll
                for (int cc = 0; cc < KC; ++cc) fma_col(S + cc * SOS, c0 + cc);
            } else {
                for (int cc = 0; cc < K - c0; ++cc) fma_col(S + cc * SOS, c0 + cc);
            }
            if (kc + 1 < nkc) {
                store_op(b ^ 1);
                if (kc + 2 < nkc) load_op(li, c0 + 2 * KC);
                else if (li + 1 < hi) load_op(li + 1, 0);
            }
            __syncthreads();  // chunk kc is read; chunk kc + 1 is in LDS
        }
    }
#pragma unroll
    for (int jj = 0; jj < CPT; ++jj) {
        const int32_t t = tgt[tc * CPT + jj];
        if (t < 0) continue;
        R *dst = nsplit == 1 ? Lx + static_cast<size_t>(t) * ldk
                             : part + (static_cast<size_t>(sp) * 8 * nparents + static_cast<size_t>(chunk * TB + tc * CPT + jj) * 8 + qt) * ldk;
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const int r = tr + 32 * i;
            if (r < K) dst[r] = sg[r] * acc[i][jj];
        }
    }
}

// ---------------------------------------------------------------------------
// FP32 M2L on v_mfma_f32_16x16x4: the same offset-grouped product as
// k_m2l_plain, a block of 4 wavefronts per (chunk of TB parents, child octant).
// A wavefront (wr, wc) owns half of the 16-row tiles and half of the 16-target
// tiles (an odd middle row tile is split by target tiles), so operator
// fragments come straight from L2 in 16-byte words that feed 4 x TB / 32
// products each, one column group ahead, and only the gathered, mirrored
// multipoles go through LDS, in rows of the targets (16-byte copies of the
// expansions; the row stride is an odd number of 16-byte words, so reads have
// no bank conflicts).  The matrix pipe is what bounds it: a product takes 32
// cycles and VALU work adds to it (both use the FP32 units), so the layout
// keeps that work small: operator addresses are uniform, a lane gathers the
// same word of every target, so its mirror signs are four registers, and the
// next offset's multipoles are on their way during the products.  FP32 FMAs
// from LDS (k_m2l_plain's form, 64 targets) ran at 58 % of the one-FMA-a-cycle
// rate; M2L per evaluation, then and now: 4M Plummer p = 12 19.1 -> 9.4 ms
// (91 TFLOP/s, 60 % of a large FP32 matrix product), 10^6 Plummer p = 12 6.1 ->
// 2.4, 2^20 uniform p = 8 2.67 -> 1.14, p = 5 1.40 -> 0.33, p = 3 0.59 -> 0.09,
// 16,384 Plummer p = 8 0.099 -> 0.070.  Blocks of 32 targets were slower at every size.
// ---------------------------------------------------------------------------
typedef float f4 __attribute__((ext_vector_type(4)));
template <int P>
struct M2lShape {
    static constexpr int K = (P + 1) * (P + 1), NT = (K + 15) / 16, NKS = (K - 16 * (NT - 1) + 3) / 4, LD = (K + 3) / 4 * 4, LD4 = LD / 4;
    static constexpr int SK = (LD4 | 1) * 4;  // LDS row stride
    static constexpr int H = NT / 2;          // whole row tiles per wavefront
    static constexpr int TPI = 64 / LD4;      // targets a wavefront gathers with one load
};
template <int P>
__global__ __launch_bounds__(256, 2) void k_m2l_f32(const int32_t *__restrict__ parents, int nparents, const int32_t *__restrict__ child,
                                                    const uint32_t *__restrict__ count, const int32_t *__restrict__ nbr27,
                                                    const f4 *__restrict__ Mx, float *__restrict__ Lx, const f4 *__restrict__ op, int nsplit,
                                                    float *__restrict__ part) {
    using S = M2lShape<P>;
    constexpr int TB = 64;                          // targets
    constexpr int NC = TB / 32;                     // 16-target tiles per wavefront
    constexpr int HX = S::H + (S::NT & 1);          // row tiles it loads
    constexpr int NG = (TB + 4 * S::TPI - 1) / (4 * S::TPI);  // 16-byte words a thread gathers
    __shared__ __align__(16) float sM[TB * S::SK];
    __shared__ int32_t s_nc[27 * TB];  // first child of parent neighbour d of target t, or -1
    __shared__ uint8_t s_nm[27 * TB];  // its non-empty children
    __shared__ int32_t tgt[TB];
    __shared__ int16_t s_o[189], s_dn[189], s_qs[189], s_live[189];
    __shared__ int s_nlive, s_cnt[3];
    const int nchunks = (nparents + TB - 1) / TB;
    const int per = nchunks * nsplit;                           // work items per XCD
    const int wi = (blockIdx.x & 7) * per + (blockIdx.x >> 3);  // XCD x takes work items [x W / 8, (x + 1) W / 8)
    if (wi >= 8 * per) return;
    const int sp = wi % nsplit, w = wi / nsplit;  // the parts of one (chunk, octant) are neighbours
    const int chunk = w >> 3, qt = w & 7;
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, quad = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wv & 1, wc = wv >> 1;
    m2l_walk(tid, 256, qt, s_o, s_dn, s_qs);
    if (tid < TB) {
        const int pi = chunk * TB + tid;
        const int32_t p = pi < nparents ? parents[pi] : -1;
        int32_t t = p >= 0 ? child[p] + qt : -1;
        if (t >= 0 && count[t] == 0) t = -1;
        tgt[tid] = t;
    }
    __syncthreads();
    for (int i = tid; i < 27 * TB; i += 256) {
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
    // this lane gathers word ch of the targets (wv + 4 u) TPI + sub
    const int sub = lane / S::LD4, ch = lane % S::LD4;
    uint32_t sg[4];  // its mirror signs
#pragma unroll
    for (int e = 0; e < 4; ++e) sg[e] = 4 * ch + e < S::K && m2l_mirror_sign(qt, 4 * ch + e) < 0 ? 0x80000000u : 0u;
    __syncthreads();
    const int nlive = s_nlive;
    const int lo = sp * nlive / nsplit, hi = (sp + 1) * nlive / nsplit;  // this block's walked offsets
    f4 acc[HX][NC], sum[HX][NC];  // the current offset's products, and the sum of the offsets before it
#pragma unroll
    for (int h = 0; h < HX; ++h)
#pragma unroll
        for (int n = 0; n < NC; ++n) sum[h][n] = f4{0, 0, 0, 0};
    // row tile h of this wavefront: wr H .. wr H + H - 1, and the last one (of an odd number) for half of the targets
    auto row_tile = [&](int h) { return h < S::H ? wr * S::H + h : S::NT - 1; };
    auto load_a = [&](int li, int j, f4 *a) {  // (uniform base, lane offset)
        const f4 *O = op + static_cast<size_t>(__builtin_amdgcn_readfirstlane(s_o[s_live[li]])) * (S::NT * S::NT * 64) + j * 64;
#pragma unroll
        for (int h = 0; h < HX; ++h) a[h] = (O + row_tile(h) * (S::NT * 64))[static_cast<unsigned>(lane)];
    };
    const float *Brow = sM + (wc * 16 * NC + col) * S::SK;
    f4 an[HX], v[NG];
    auto gather = [&](int li) {  // this thread's words of the multipoles of walked offset li
        const int st = s_live[li], dn = __builtin_amdgcn_readfirstlane(s_dn[st]) * TB, qs = __builtin_amdgcn_readfirstlane(s_qs[st]);
#pragma unroll
        for (int u = 0; u < NG; ++u) {
            v[u] = f4{0, 0, 0, 0};
            if constexpr (S::TPI == 1) {  // one target: its lookups are uniform
                const int t = dn + wv + 4 * u;
                const int cell = __builtin_amdgcn_readfirstlane(s_nc[t]) + qs;
                if ((__builtin_amdgcn_readfirstlane(s_nm[t]) >> qs) & 1)
                    if (lane < S::LD4) v[u] = (Mx + static_cast<size_t>(cell) * S::LD4)[static_cast<unsigned>(lane)];
            } else {
                const int t = (wv + 4 * u) * S::TPI + sub;
                if (sub < S::TPI && t < TB && ((s_nm[dn + t] >> qs) & 1)) v[u] = Mx[static_cast<size_t>(s_nc[dn + t] + qs) * S::LD4 + ch];
            }
        }
    };
    if (hi > lo) {
        load_a(lo, 0, an);
        gather(lo);
    }
    for (int li = lo; li < hi; ++li) {
#pragma unroll
        for (int u = 0; u < NG; ++u) {
            const int t = (wv + 4 * u) * S::TPI + sub;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[u][e] = __uint_as_float(__float_as_uint(v[u][e]) ^ sg[e]);
            if (sub < S::TPI && t < TB) *reinterpret_cast<f4 *>(sM + t * S::SK + 4 * ch) = v[u];
        }
        if (li + 1 < hi) gather(li + 1);  // on its way during the products
        __syncthreads();  // the multipoles of this offset are in LDS
        // the products of one column group; the offset's first ones start its sums
        auto group = [&](const f4 *a, const f4 *b, int nk, auto first) {
            const f4 zero = {0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i >= nk) break;
                const bool start = decltype(first)::value && i == 0;
#pragma unroll
                for (int h = 0; h < S::H; ++h)
#pragma unroll
                    for (int n = 0; n < NC; ++n) acc[h][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[h][i], b[n][i], start ? zero : acc[h][n], 0, 0, 0);
                if constexpr (S::NT & 1)
                    acc[S::H][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[S::H][i], wr ? b[1][i] : b[0][i], start ? zero : acc[S::H][0], 0, 0, 0);
            }
        };
        auto full = [&](int j, auto first) {
            f4 a[HX], b[NC];
#pragma unroll
            for (int h = 0; h < HX; ++h) a[h] = an[h];
            load_a(li, j + 1, an);
#pragma unroll
            for (int n = 0; n < NC; ++n) b[n] = *reinterpret_cast<const f4 *>(Brow + 16 * n * S::SK + 16 * j + 4 * quad);
            group(a, b, 4, first);
        };
        if constexpr (S::NT > 1) full(0, std::true_type{});
#pragma unroll 2
        for (int j = 1; j + 1 < S::NT; ++j) full(j, std::false_type{});
        {  // the last column group
            f4 a[HX], b[NC];
#pragma unroll
            for (int h = 0; h < HX; ++h) a[h] = an[h];
            if (li + 1 < hi) load_a(li + 1, 0, an);
#pragma unroll
            for (int n = 0; n < NC; ++n)
#pragma unroll
                for (int i = 0; i < S::NKS; ++i) b[n][i] = Brow[16 * n * S::SK + 16 * (S::NT - 1) + S::NKS * quad + i];
            group(a, b, S::NKS, std::bool_constant<S::NT == 1>{});
        }
        // offset by offset: shorter sums, so less rounding (RMS error of the locals against FP64 at p = 3 and 5:
        // 1.1e-7 and 1.6e-7 in one sum, as in k_m2l_plain's form, 0.8e-7 and 1.0e-7 here)
#pragma unroll
        for (int h = 0; h < HX; ++h)
#pragma unroll
            for (int n = 0; n < NC; ++n) sum[h][n] += acc[h][n];
        __syncthreads();  // every wavefront has read the multipoles
    }
    // D: lane holds rows 4 quad .. 4 quad + 3 of a tile for target col
    auto put = [&](int tile, int n, f4 v) {
        const int ti = (wc * NC + n) * 16 + col, r0 = 16 * tile + 4 * quad;
        const int32_t t = tgt[ti];
        if (t < 0 || r0 >= S::LD) return;
        float *dst = nsplit == 1 ? Lx + static_cast<size_t>(t) * S::LD
                                 : part + (static_cast<size_t>(sp) * 8 * nparents + static_cast<size_t>(chunk * TB + ti) * 8 + qt) * S::LD;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (r0 + e < S::K && m2l_mirror_sign(qt, r0 + e) < 0) v[e] = -v[e];
        *reinterpret_cast<f4 *>(dst + r0) = v;
    };
#pragma unroll
    for (int h = 0; h < S::H; ++h)
#pragma unroll
        for (int n = 0; n < NC; ++n) put(wr * S::H + h, n, sum[h][n]);
    if constexpr (S::NT & 1) put(S::NT - 1, wr, sum[S::H][0]);
}

// ---------------------------------------------------------------------------
// FP32 M2M (UP, solver_ref.hpp:196-197) and L2L (solver_ref.hpp:217-218) of one tree
// level on v_mfma_f32_16x16x4.  A block takes one 16-row tile of 16 TN parents, a
// wavefront each octant q: M2M multiplies child q's multipoles and the block adds the 8
// products in octant order, L2L adds its product to child q's locals.  The operands of
// four column groups at a time come from L2 straight into registers, without
// LDS, and the column groups that the operator's triangle leaves empty are skipped
// (M2M: degrees above the rows' last, L2L: below their first).  Products go
// through the columns in order, so the sums are those of an FMA per column.
// Most levels are small, and bound by the latency of one pass: a lane per operator row
// with one column after the other (k_m2m_wide's form) took up to 43 us a level, where
// this takes 6 to 13.  L2L per evaluation, then and now: 10^6 Plummer p = 12 301 -> 132 us,
// 64,000 p = 8 50 -> 30, 2^20 uniform p = 8 62 -> 41; RK4 steps 17.1 -> 16.3, 2.49 -> 2.39 and
// 7.92 -> 7.73 ms.
// ---------------------------------------------------------------------------
template <int P, int TN, bool UP>
__global__ __launch_bounds__(512) void k_ml_f32(const int32_t *__restrict__ ids, int n, const int32_t *__restrict__ child,
                                                const uint32_t *__restrict__ count, const f4 *__restrict__ op, float *__restrict__ X) {
    using S = M2lShape<P>;
    constexpr int NB = 4;  // column groups in flight
    const int lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
    const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rt = blockIdx.x % S::NT, p0 = blockIdx.x / S::NT * 16 * TN;
    int32_t cell[TN], par[TN];  // child q (-1: empty or none) and parent of column 16 t + col
    const float *src[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        const int i = p0 + 16 * t + col;
        par[t] = i < n ? ids[i] : -1;
        cell[t] = par[t] >= 0 ? child[par[t]] + q : -1;
        if (cell[t] >= 0 && count[cell[t]] == 0) cell[t] = -1;
        const int32_t from = UP || cell[t] < 0 ? cell[t] : par[t];
        src[t] = from >= 0 ? X + static_cast<size_t>(from) * S::LD : nullptr;
    }
    int g0 = 0, g1 = S::NT;  // column groups that hold something
    {
        const int r = UP ? min(16 * rt + 15, S::K - 1) : 16 * rt;
        int j = 0;  // degree of row r
        while ((j + 1) * (j + 1) <= r) ++j;
        if (UP)
            g1 = ((j + 1) * (j + 1) + 15) / 16;
        else
            g0 = j * j / 16;
    }
    const f4 *A = op + (static_cast<size_t>(UP ? q : 8 + q) * S::NT + rt) * S::NT * 64;
    const f4 zero = {0, 0, 0, 0};
    f4 acc[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t) acc[t] = zero;
    for (int g = g0; g < g1; g += NB) {
        f4 a[NB], b[NB][TN];
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            a[u] = g + u < g1 ? A[(g + u) * 64 + lane] : zero;
#pragma unroll
            for (int t = 0; t < TN; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int k = 16 * (g + u) + 4 * i + quad;
                    b[u][t][i] = g + u < g1 && src[t] && k < S::K ? src[t][k] : 0.0f;
                }
        }
#pragma unroll
        for (int u = 0; u < NB; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int t = 0; t < TN; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i], b[u][t][i], acc[t], 0, 0, 0);
    }
    // lane: rows 16 rt + 4 quad .. + 3 of column 16 t + col
    const int w = 4 * rt + quad;
    if constexpr (UP) {
        __shared__ f4 s_acc[8][TN][64];
#pragma unroll
        for (int t = 0; t < TN; ++t) s_acc[q][t][lane] = acc[t];
        __syncthreads();
        if (q < TN) {  // wavefront t adds the octants' products of its 16 parents
            f4 sum = s_acc[0][q][lane];
#pragma unroll
            for (int o = 1; o < 8; ++o) sum += s_acc[o][q][lane];
            const int i = p0 + 16 * q + col;
            if (i < n && w < S::LD4) reinterpret_cast<f4 *>(X)[static_cast<size_t>(ids[i]) * S::LD4 + w] = sum;
        }
    } else {
        if (w < S::LD4) {
#pragma unroll
            for (int t = 0; t < TN; ++t)
                if (cell[t] >= 0) reinterpret_cast<f4 *>(X)[static_cast<size_t>(cell[t]) * S::LD4 + w] += acc[t];
        }
    }
}

// The nsplit partial sums of each non-empty M2L target into its local
// expansion, in part order (one thread per target slot and coefficient).
template <class R>
__global__ __launch_bounds__(256) void k_m2l_sum(const int32_t *__restrict__ parents, int nparents, const int32_t *__restrict__ child,
                                                 const uint32_t *__restrict__ count, int nsplit, const R *__restrict__ part, R *__restrict__ Lx,
                                                 int K, int ldk) {
    const int64_t i = blockIdx.x * 256ll + threadIdx.x;
    if (i >= static_cast<int64_t>(8) * nparents * K) return;
    const int64_t slot = i / K;
    const int r = static_cast<int>(i % K);
    const int32_t t = child[parents[slot >> 3]] + static_cast<int32_t>(slot & 7);
    if (count[t] == 0) return;
    const size_t stride = static_cast<size_t>(8) * nparents * ldk;
    R v = part[static_cast<size_t>(slot) * ldk + r];
#pragma unroll 8
    for (int q = 1; q < nsplit; ++q) v += part[q * stride + static_cast<size_t>(slot) * ldk + r];
    Lx[static_cast<size_t>(t) * ldk + r] = v;
}

// ---------------------------------------------------------------------------
// L2P: one thread per particle of a leaf; the R_n^m recurrence feeds the
// potential, d/dz and (d/dx - i d/dy) directly, so no table is stored.
// ---------------------------------------------------------------------------
// Recurrence and ladder coefficients as functions of (n, m): with p a template
// parameter and the loops unrolled they fold to immediates (P2M, whose lanes have
// different orders m, reads the first three from the __constant__ tables).  The last
// three are the gradient's ladder.
__device__ __forceinline__ double k_diag(int m) { return -sqrt((2.0 * m - 1) / (2.0 * m)); }
__device__ __forceinline__ double k_r1(int n, int m) { return (2.0 * n - 1) / sqrt(static_cast<double>(n - m) * (n + m)); }
__device__ __forceinline__ double k_r2(int n, int m) { return sqrt(static_cast<double>(n + m - 1) * (n - m - 1) / (static_cast<double>(n - m) * (n + m))); }
__device__ __forceinline__ double k_lz(int l, int m) { return m <= l ? sqrt(static_cast<double>(l + m) * (l - m)) : 0.0; }
__device__ __forceinline__ double k_la(int l, int m) { return m <= l ? sqrt(static_cast<double>(l + m) * (l + m - 1)) : 0.0; }
__device__ __forceinline__ double k_lb(int l, int m) { return m + 1 <= l ? sqrt(static_cast<double>(l - m) * (l - m - 1)) : 0.0; }

// The P2P's results and the caller's arrays, for L2P to add to.
template <class R>
struct Near {
    const Quad<R> *acc;                 // sums of the leaves with one work item, times G
    const Quad<R> *part;                // rows of partial sums of the others
    const uint32_t *nchunk, *item_off;  // per leaf: rows (1: none) of whole 16-particle tiles, first tile
    R G;
    const uint32_t *perm;  // caller's index of a sorted particle
    R *a;                  // accelerations in the caller's order
    double *pot;           // potentials, or nullptr
};

// A block per leaf, a lane per particle: the near field (partial sums of split
// leaves added in chunk order, the same order every run), the far field, and the sum
// to the caller's place.  Bound by VALU issue, and small trees by launches: the
// sums of split leaves and the way back to the caller's order were two more
// kernels, 16 bytes a particle written and read again for each. RK4 step of
// 2^20 uniform particles 7.74 -> 7.66 ms, 4M Plummer 36.5 -> 36.15, 16384 FP64 1.27 -> 1.24.
// flag: only the leaves where it is `want`.
template <class R, int P, bool POT>
__global__ __launch_bounds__(64) void k_l2p(const int32_t *__restrict__ leaves, const int8_t *__restrict__ level, const uint32_t *__restrict__ start,
                                            const uint32_t *__restrict__ count, const double *__restrict__ bmin, const double *__restrict__ bmax,
                                            const double4 *__restrict__ xs64, double wx0, int ldk, const R *__restrict__ Lx, double gscale, Near<R> near,
                                            const uint8_t *__restrict__ flag, bool want) {
    __shared__ R sl[MAXK];
    if (flag && (flag[blockIdx.x] != 0) != want) return;  // the closure's fallback leaves, or the others
    const int32_t c = leaves[blockIdx.x];
    const bool far = level[c] >= 2;  // solver_ref.hpp:220-221
    constexpr int K = (P + 1) * (P + 1);
    if (far)
        for (int i = threadIdx.x; i < K; i += 64) sl[i] = Lx[static_cast<size_t>(c) * ldk + i];
    __syncthreads();
    const uint32_t s = start[c], cnt = count[c], nch = near.nchunk[blockIdx.x];
    const Quad<R> *part = near.part + static_cast<size_t>(nch > 1 ? near.item_off[blockIdx.x] : 0) * 16;
    const uint32_t pstride = (cnt + 15) / 16 * 16;
    const double w = ldexp(wx0, -level[c]);
    const double iw = 1.0 / w;
    const double cx = (bmin[3 * c] + bmax[3 * c]) / 2, cy = (bmin[3 * c + 1] + bmax[3 * c + 1]) / 2, cz = (bmin[3 * c + 2] + bmax[3 * c + 2]) / 2;
    for (uint32_t i = threadIdx.x; i < cnt; i += 64) {
        const uint32_t k = s + i;
        const uint32_t at = near.perm[k];
        const double4 xm = xs64[k];
        Quad<R> v;
        if (nch < 2) {
            v = near.acc[k];
        } else {
            v.x = v.y = v.z = v.w = 0;
#pragma unroll 8
            for (uint32_t q = 0; q < nch; ++q) {
                const Quad<R> u = part[static_cast<size_t>(q) * pstride + i];
                v.x += u.x;
                v.y += u.y;
                v.z += u.z;
                v.w += u.w;
            }
            v.x *= near.G, v.y *= near.G, v.z *= near.G;
        }
        auto store = [&] {
            near.a[3ll * at] = v.x;
            near.a[3ll * at + 1] = v.y;
            near.a[3ll * at + 2] = v.z;
            if (POT) near.pot[at] = static_cast<double>(v.w);
        };
        if (!far) {
            store();
            continue;
        }
        // read the local coefficients from LDS inside the loop rather than hold all of them in registers
        int z0 = 0;
        asm volatile("" : "+v"(z0));
        const R *slv = sl + z0;
        const R x = static_cast<R>((xm.x - cx) * iw), y = static_cast<R>((xm.y - cy) * iw), z = static_cast<R>((xm.z - cz) * iw);
        const R r2 = x * x + y * y + z * z;
        R phi = 0, gz = 0, gre = 0, gim = 0;  // potential, d/dz, (d/dx - i d/dy)
        R dre = 1, dim = 0;
#pragma unroll
        for (int m = 0; m <= P; ++m) {
            if (m > 0) {
                const R d = static_cast<R>(k_diag(m));
                const R nre = d * (x * dre - y * dim), nim = d * (x * dim + y * dre);
                dre = nre;
                dim = nim;
            }
            R are = 0, aim = 0, cre = dre, cim = dim;  // R_{n-2}^m, R_n^m
#pragma unroll
            for (int n = m; n <= P; ++n) {
                if (n > m) {
                    const R c1 = static_cast<R>(k_r1(n, m)), c2 = static_cast<R>(k_r2(n, m));
                    const R nre = c1 * z * cre - c2 * r2 * are, nim = c1 * z * cim - c2 * r2 * aim;
                    are = cre;
                    aim = cim;
                    cre = nre;
                    cim = nim;
                }
                // potential: sum L_n^0 R_n^0 + 2 Re(L_n^m R_n^m)
                if (!POT)
                    ;
                else if (m == 0)
                    phi += slv[kidx_re(n, 0)] * cre;
                else
                    phi += 2 * (slv[kidx_re(n, m)] * cre - slv[kidx_im(n, m)] * cim);
                if (n + 1 <= P) {
                    const int l = n + 1;  // R_n^m enters the derivatives of degree-l terms
                    const R lz = static_cast<R>(k_lz(l, m));
                    if (m == 0)
                        gz += slv[kidx_re(l, 0)] * lz * cre;
                    else
                        gz += 2 * lz * (slv[kidx_re(l, m)] * cre - slv[kidx_im(l, m)] * cim);
                    {  // -sqrt((l+m+1)(l+m)) L_l^{m+1} R_n^m
                        const R la = static_cast<R>(k_la(l, m + 1));
                        const R Lre = slv[kidx_re(l, m + 1)], Lim = slv[kidx_im(l, m + 1)];
                        gre -= la * (Lre * cre - Lim * cim);
                        gim -= la * (Lre * cim + Lim * cre);
                    }
                    if (m >= 1) {  // sqrt((l-m+1)(l-m)) conj(L_l^{m-1} R_n^m), with Re(L_l^0) for m = 1
                        const R lb = static_cast<R>(k_lb(l, m - 1));
                        const R Lre = slv[kidx_re(l, m - 1)], Lim = (m - 1) == 0 ? R(0) : slv[kidx_im(l, m - 1)];
                        gre += lb * (Lre * cre - Lim * cim);
                        gim -= lb * (Lre * cim + Lim * cre);
                    }
                }
            }
        }
        const R gs = static_cast<R>(gscale * iw * iw);
        v.x += gs * gre;
        v.y -= gs * gim;
        v.z += gs * gz;
        if (POT) v.w += static_cast<R>(iw) * phi;
        store();
    }
}

template <class R>
Near<R> near_of(Ctx &c, const DevBuf<R> &acc, const DevBuf<R> &part, DevBuf<R> &a, bool potential) {
    const size_t n = static_cast<size_t>(std::max<int64_t>(1, c.n));
    a.ensure(3 * n);
    if (potential) c.pot64.ensure(n);
    return {reinterpret_cast<const Quad<R> *>(acc.p), reinterpret_cast<const Quad<R> *>(part.p), c.p2p_nchunk, c.p2p_item_off,
            static_cast<R>(c.G), c.perm, a.p, potential ? c.pot64.p : nullptr};
}

template <class R>
struct Bufs;
template <>
struct Bufs<double> {
    static double *M(Ctx &c) { return c.M64; }
    static double *L(Ctx &c) { return c.L64; }
    static Near<double> near(Ctx &c, bool potential) { return near_of<double>(c, c.as64, c.p2p_part64, c.acc64, potential); }
    static void ensure(Ctx &c, size_t nc) {
        c.M64.ensure(nc * c.ldk + 16);
        c.L64.ensure(nc * c.ldk + 16);
    }
};
template <>
struct Bufs<float> {
    static float *M(Ctx &c) { return c.M32; }
    static float *L(Ctx &c) { return c.L32; }
    static Near<float> near(Ctx &c, bool potential) { return near_of<float>(c, c.as32, c.p2p_part32, c.acc32, potential); }
    static void ensure(Ctx &c, size_t nc) {
        c.M32.ensure(nc * c.ldk + 16);
        c.L32.ensure(nc * c.ldk + 16);
    }
};

// One parent per 1024-thread block, for the small levels near the root: the
// (child q, row r) items are spread over the threads; M2M then adds the 8
// children's partial rows through LDS.
__global__ __launch_bounds__(1024) void k_m2m_wide(const int32_t *__restrict__ ids, const int32_t *__restrict__ child, const uint32_t *__restrict__ count,
                                                   const double *__restrict__ op, int K, int ldk, double *__restrict__ M) {
    __shared__ double cm[8 * MAXK];
    __shared__ double part[8 * MAXK];
    const int32_t P = ids[blockIdx.x];
    const int32_t cb = child[P];
    for (int i = threadIdx.x; i < 8 * K; i += 1024) {
        const int q = i / K, col = i % K;
        cm[i] = count[cb + q] ? M[static_cast<size_t>(cb + q) * ldk + col] : double(0);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 8 * K; i += 1024) {
        const int q = i / K, r = i % K;
        int j = 0;
        while ((j + 1) * (j + 1) <= r) ++j;
        const double *ocol = op + static_cast<size_t>(q) * K * K + r;
        double sum = 0;
        for (int col = 0; col < (j + 1) * (j + 1); ++col) sum += ocol[static_cast<size_t>(col) * K] * cm[q * K + col];
        part[i] = sum;
    }
    __syncthreads();
    for (int r = threadIdx.x; r < K; r += 1024) {
        double sum = 0;
        for (int q = 0; q < 8; ++q) sum += part[q * K + r];  // children in order
        M[static_cast<size_t>(P) * ldk + r] = sum;
    }
    for (int i = K + threadIdx.x; i < ldk; i += 1024) M[static_cast<size_t>(P) * ldk + i] = double(0);
}

__global__ __launch_bounds__(1024) void k_l2l_wide(const int32_t *__restrict__ ids, const int32_t *__restrict__ child, const uint32_t *__restrict__ count,
                                                   const double *__restrict__ op, int K, int ldk, double *__restrict__ L) {
    __shared__ double pl[MAXK];
    const int32_t P = ids[blockIdx.x];
    const int32_t cb = child[P];
    for (int i = threadIdx.x; i < K; i += 1024) pl[i] = L[static_cast<size_t>(P) * ldk + i];
    __syncthreads();
    for (int i = threadIdx.x; i < 8 * K; i += 1024) {
        const int q = i / K, r = i % K;
        if (!count[cb + q]) continue;
        int j = 0;
        while ((j + 1) * (j + 1) <= r) ++j;
        const double *ocol = op + static_cast<size_t>(8 + q) * K * K + r;
        double sum = 0;
        for (int col = j * j; col < K; ++col) sum += ocol[static_cast<size_t>(col) * K] * pl[col];
        L[static_cast<size_t>(cb + q) * ldk + r] += sum;
    }
}

inline int pick_pb(int64_t nparents, int maxpb) {
    int pb = 1;
    while (pb < maxpb && nparents >= static_cast<int64_t>(pb) * 2 * 512) pb *= 2;
    return pb;
}

template <int P, bool UP>
void ml_f32_launch(Ctx &c, const int32_t *ids, int n) {
    using S = M2lShape<P>;
    if (c.ldk != S::LD) throw Error(1, "FP32 M2M and L2L: the coefficient stride must be K rounded up to 4");
    const TreeDev &t = c.t;
    const f4 *op = reinterpret_cast<const f4 *>(c.op32.p);
    float *X = UP ? c.M32.p : c.L32.p;
    // two tiles of parents share an operator fragment where that leaves a block for every CU
    if (ceil_div(n, 32) * S::NT >= c.ncu)
        k_ml_f32<P, 2, UP><<<ceil_div(n, 32) * S::NT, 512, 0, c.stream>>>(ids, n, t.child, t.count, op, X);
    else
        k_ml_f32<P, 1, UP><<<ceil_div(n, 16) * S::NT, 512, 0, c.stream>>>(ids, n, t.child, t.count, op, X);
}

template <bool UP>
void ml_f32_level(Ctx &c, const int32_t *ids, int n) {
    switch (c.p) {
    case 1: ml_f32_launch<1, UP>(c, ids, n); break;
    case 2: ml_f32_launch<2, UP>(c, ids, n); break;
    case 3: ml_f32_launch<3, UP>(c, ids, n); break;
    case 4: ml_f32_launch<4, UP>(c, ids, n); break;
    case 5: ml_f32_launch<5, UP>(c, ids, n); break;
    case 6: ml_f32_launch<6, UP>(c, ids, n); break;
    case 7: ml_f32_launch<7, UP>(c, ids, n); break;
    case 8: ml_f32_launch<8, UP>(c, ids, n); break;
    case 9: ml_f32_launch<9, UP>(c, ids, n); break;
    case 10: ml_f32_launch<10, UP>(c, ids, n); break;
    case 11: ml_f32_launch<11, UP>(c, ids, n); break;
    case 12: ml_f32_launch<12, UP>(c, ids, n); break;
    default: throw Error(1, "M2M and L2L support 1 <= p <= 12");
    }
}

// M2M (up) or L2L of the internal cells of one level
void ml_level(Ctx &c, const int32_t *ids, int64_t n, bool up) {
    const TreeDev &t = c.t;
    if (c.prec == 2) {  // on the matrix cores, with split operands
        ml_split_level(c, ids, n, up);
        return;
    }
    if (c.prec == 1) {
        up ? ml_f32_level<true>(c, ids, static_cast<int>(n)) : ml_f32_level<false>(c, ids, static_cast<int>(n));
        return;
    }
    if (n < 1024) {  // few parents: one wide block each
        if (up)
            k_m2m_wide<<<static_cast<unsigned>(n), 1024, 0, c.stream>>>(ids, t.child, t.count, c.op64, c.K, c.ldk, c.M64);
        else
            k_l2l_wide<<<static_cast<unsigned>(n), 1024, 0, c.stream>>>(ids, t.child, t.count, c.op64, c.K, c.ldk, c.L64);
        return;
    }
#define VG_M2M(PB_) k_m2m<PB_><<<ceil_div(n, PB_), 256, 0, c.stream>>>(ids, static_cast<int>(n), t.child, t.count, c.op64, c.K, c.ldk, c.M64)
#define VG_L2L(PB_) k_l2l<PB_><<<ceil_div(n, PB_), 256, 0, c.stream>>>(ids, static_cast<int>(n), t.child, t.count, c.op64, c.K, c.ldk, c.L64)
    const int pb = pick_pb(n, up ? 8 : 16);  // M2M: 8 children x PB staged expansions in LDS
    if (pb == 1) up ? VG_M2M(1) : VG_L2L(1);
    else if (pb == 2) up ? VG_M2M(2) : VG_L2L(2);
    else if (pb == 4) up ? VG_M2M(4) : VG_L2L(4);
    else if (pb == 8) up ? VG_M2M(8) : VG_L2L(8);
    else VG_L2L(16);
#undef VG_M2M
#undef VG_L2L
}

template <class R>
void upward_t(Ctx &c) {
    TreeDev &t = c.t;
    Bufs<R>::ensure(c, t.ncells);
    if (c.prec == 2) c.msplit.ensure(static_cast<size_t>(t.ncells) * 2 * c.ldk);
    uint16_t *ms = c.prec == 2 ? c.msplit.p : nullptr;
    const double wx0 = t.box[3] - t.box[0];
    if (t.nleaves) {
#define VG_P2M(P_)                                                                                                                          \
    k_p2m<R, P_><<<ceil_div(t.nleaves, 4), 256, 0, c.stream>>>(t.leaf_ids, static_cast<int>(t.nleaves), t.level, t.start, t.count, t.bmin, \
                                                               t.bmax, c.xs64, wx0, c.K, c.ldk, Bufs<R>::M(c), ms)
        switch (c.p) {
            case 1: VG_P2M(1); break;
            case 2: VG_P2M(2); break;
            case 3: VG_P2M(3); break;
            case 4: VG_P2M(4); break;
            case 5: VG_P2M(5); break;
            case 6: VG_P2M(6); break;
            case 7: VG_P2M(7); break;
            case 8: VG_P2M(8); break;
            case 9: VG_P2M(9); break;
            case 10: VG_P2M(10); break;
            case 11: VG_P2M(11); break;
            case 12: VG_P2M(12); break;
            default: throw Error(1, "P2M supports 1 <= p <= 12");
        }
#undef VG_P2M
    }
    for (int d = t.depth; d >= 2; --d) {
        const int64_t a = t.int_off[d], b = t.int_off[d + 1];
        if (b > a) ml_level(c, t.int_ids.p + a, b - a, true);
    }
    VG_LAUNCH_CHECK();
}

template <int TB, int RPT>
void m2l_plain_launch(Ctx &c, const int32_t *parents, int np, unsigned grid, int nsplit, double *part) {
    constexpr int KC = 8;
    const size_t lds = (static_cast<size_t>(c.K) * (TB + 2) + 2 * KC * (32 * RPT + 1)) * sizeof(double);
    // dynamic LDS above 64 KiB is allowed per kernel and device, here for the
    // largest K of this RPT (set once per device, under a lock: contexts of
    // different host threads may launch concurrently)
    static std::mutex mu;
    static uint64_t done = 0;  // bit d: set on device d
    {
        std::lock_guard<std::mutex> lock(mu);
        const uint64_t bit = c.device < 64 ? (1ull << c.device) : 0;
        if (!bit || !(done & bit)) {
            const size_t cap = (static_cast<size_t>(32 * RPT) * (TB + 2) + 2 * KC * (32 * RPT + 1)) * sizeof(double);
            VG_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_m2l_plain<TB, RPT>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       static_cast<int>(cap)));
            done |= bit;
        }
    }
    const TreeDev &t = c.t;
    k_m2l_plain<TB, RPT><<<grid * nsplit, 256, lds, c.stream>>>(parents, np, t.child, t.count, t.nbr27, c.M64, c.L64, c.op64, c.K, c.ldk, nsplit, part);
    if (nsplit > 1)
        k_m2l_sum<double><<<ceil_div(static_cast<size_t>(8) * np * c.K, 256), 256, 0, c.stream>>>(parents, np, t.child, t.count, nsplit, part, c.L64,
                                                                                               c.K, c.ldk);
    VG_LAUNCH_CHECK();
}

template <int TB>
void m2l_plain_rows(Ctx &c, const int32_t *parents, int np) {
    const int rpt = ceil_div(c.K, 32);
    const unsigned grid = 8 * ceil_div(np, TB);  // one block per (parent chunk, child octant)
    // under four blocks per CU: the walked offsets of a (chunk, octant) are cut
    // into parts, one block each (at most 32 parts, so a part keeps about six of
    // the at most 189 offsets), and a second kernel adds the partial sums (the
    // 16k Plummer sphere at p = 4: 40 blocks, 26 parts, 0.46 -> 0.05 ms)
    int nsplit = 1;
    if (c.ncu > 0 && grid < 4u * static_cast<unsigned>(c.ncu)) nsplit = std::min<int>(32, static_cast<int>(ceil_div(4 * c.ncu, grid)));
    double *part = nullptr;
    if (nsplit > 1) {
        c.m2l_part.ensure(static_cast<size_t>(nsplit) * 8 * np * c.ldk * sizeof(double));
        part = reinterpret_cast<double *>(c.m2l_part.p);
    }
    switch (rpt) {
    case 1: m2l_plain_launch<TB, 1>(c, parents, np, grid, nsplit, part); break;
    case 2: m2l_plain_launch<TB, 2>(c, parents, np, grid, nsplit, part); break;
    case 3: m2l_plain_launch<TB, 3>(c, parents, np, grid, nsplit, part); break;
    case 4: m2l_plain_launch<TB, 4>(c, parents, np, grid, nsplit, part); break;
    case 5: m2l_plain_launch<TB, 5>(c, parents, np, grid, nsplit, part); break;
    case 6: m2l_plain_launch<TB, 6>(c, parents, np, grid, nsplit, part); break;
    default: throw std::runtime_error("plain M2L: expansion order out of range");
    }
}

template <int P>
void m2l_f32_launch(Ctx &c, const int32_t *parents, int np) {
    const unsigned grid = 8 * ceil_div(np, 64);
    const int nsplit = m2l_parts(grid, c.ncu);
    float *part = m2l_part_sums(c, np, nsplit);
    if (c.ldk != M2lShape<P>::LD) throw Error(1, "FP32 M2L: the coefficient stride must be K rounded up to 4");
    const TreeDev &t = c.t;
    k_m2l_f32<P><<<grid * nsplit, 256, 0, c.stream>>>(parents, np, t.child, t.count, t.nbr27, reinterpret_cast<const f4 *>(c.M32.p), c.L32.p,
                                                          reinterpret_cast<const f4 *>(c.opfrag.p), nsplit, part);
    VG_LAUNCH_CHECK();
    m2l_add_parts(c, parents, np, nsplit, part);
}

void m2l_f32_list(Ctx &c, const int32_t *parents, int np) {
    if (np <= 0) return;
    switch (c.p) {
    case 1: m2l_f32_launch<1>(c, parents, np); break;
    case 2: m2l_f32_launch<2>(c, parents, np); break;
    case 3: m2l_f32_launch<3>(c, parents, np); break;
    case 4: m2l_f32_launch<4>(c, parents, np); break;
    case 5: m2l_f32_launch<5>(c, parents, np); break;
    case 6: m2l_f32_launch<6>(c, parents, np); break;
    case 7: m2l_f32_launch<7>(c, parents, np); break;
    case 8: m2l_f32_launch<8>(c, parents, np); break;
    case 9: m2l_f32_launch<9>(c, parents, np); break;
    case 10: m2l_f32_launch<10>(c, parents, np); break;
    case 11: m2l_f32_launch<11>(c, parents, np); break;
    case 12: m2l_f32_launch<12>(c, parents, np); break;
    default: throw Error(1, "M2L supports 1 <= p <= 12");
    }
}

// FP64: 32 targets per block, half of that when this leaves fewer than four
// blocks per CU (twice the blocks keep more wavefronts in flight per CU).
void m2l_f64_list(Ctx &c, const int32_t *parents, int np) {
    if (np <= 0) return;
    if (8 * static_cast<int64_t>(ceil_div(np, 32)) < 4 * static_cast<int64_t>(c.ncu))
        m2l_plain_rows<16>(c, parents, np);
    else
        m2l_plain_rows<32>(c, parents, np);
}

template <class R>
void l2p_t(Ctx &c, bool potential, const uint8_t *flag, bool want) {
    const TreeDev &t = c.t;
    const double wx0 = t.box[3] - t.box[0];
    const double gscale = (c.flags & 1u) ? 1.0 : c.G;
    const int64_t n = t.nleaves;
    if (!n) return;
    const Near<R> near = Bufs<R>::near(c, potential);
    const double4 *xs = reinterpret_cast<const double4 *>(c.xs64.p);
    const unsigned grid = static_cast<unsigned>(n);
#define VG_L2P(P_)                                                                                                                              \
    (potential ? k_l2p<R, P_, true> : k_l2p<R, P_, false>)<<<grid, 64, 0, c.stream>>>(t.leaf_ids, t.level, t.start, t.count, t.bmin, t.bmax, xs, \
                                                                                     wx0, c.ldk, Bufs<R>::L(c), gscale, near, flag, want)
    switch (c.p) {
        case 1: VG_L2P(1); break;
        case 2: VG_L2P(2); break;
        case 3: VG_L2P(3); break;
        case 4: VG_L2P(4); break;
        case 5: VG_L2P(5); break;
        case 6: VG_L2P(6); break;
        case 7: VG_L2P(7); break;
        case 8: VG_L2P(8); break;
        case 9: VG_L2P(9); break;
        case 10: VG_L2P(10); break;
        case 11: VG_L2P(11); break;
        case 12: VG_L2P(12); break;
        default: throw Error(1, "L2P supports 1 <= p <= 12");
    }
#undef VG_L2P
    VG_LAUNCH_CHECK();
}

template <class R>
void downward_t(Ctx &c, bool potential) {
    TreeDev &t = c.t;
    for (int d = 2; d < t.depth; ++d) {  // parents at level d >= 2 feed children at level >= 3
        const int64_t a = t.int_off[d], b = t.int_off[d + 1];
        if (b > a) ml_level(c, t.int_ids.p + a, b - a, false);
    }
    join_p2p(c);  // L2P adds to the P2P accelerations
    bool fallback = false;
    if constexpr (sizeof(R) == 4) {
        if (c.cl.on) {
            closure_apply(c);                         // learned correction of the leaf locals before L2P
            fallback = closure_fallback_prepare(c);   // order-p_hi locals where the estimate exceeds the bound
        }
    }
    l2p_t<R>(c, potential, fallback ? c.cl.flag.p : nullptr, false);
    if constexpr (sizeof(R) == 4) {
        if (fallback) closure_fallback_l2p(c, potential);
    }
}

}  // namespace

void m2l_split_operators(Ctx &c);

// The tables live in each device's constant memory: upload them once per
// device (the caller has made the context's device current).
void fmm_constants_init() {
    static std::mutex mu;
    static std::vector<bool> done;
    int dev = 0;
    VG_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    if (static_cast<size_t>(dev) < done.size() && done[static_cast<size_t>(dev)]) return;
    std::vector<double> A((AL + 1) * AW, 0.0);
    for (int n = 0; n <= AL; ++n)
        for (int m = -n; m <= n; ++m) {
            const int am = m < 0 ? -m : m;
            double d = 1;
            for (int i = n - am + 1; i <= n + am; ++i) d *= i;
            d = std::sqrt(d);
            for (int i = 1; i <= n - am; ++i) d *= i;
            A[n * AW + AL + m] = (n % 2 == 0 ? 1.0 : -1.0) / d;  // fmm.hpp:201-221
        }
    std::vector<double> diag(MAXP + 1, 0), r1((MAXP + 1) * (MAXP + 1), 0), r2((MAXP + 1) * (MAXP + 1), 0);
    for (int m = 1; m <= MAXP; ++m) diag[m] = -std::sqrt((2.0 * m - 1) / (2.0 * m));
    for (int n = 1; n <= MAXP; ++n)
        for (int m = 0; m < n; ++m) {
            r1[n * (MAXP + 1) + m] = (2.0 * n - 1) / std::sqrt(static_cast<double>(n - m) * (n + m));
            r2[n * (MAXP + 1) + m] = std::sqrt(static_cast<double>(n + m - 1) * (n - m - 1) / (static_cast<double>(n - m) * (n + m)));
        }
    VG_HIP(hipMemcpyToSymbol(HIP_SYMBOL(cA), A.data(), A.size() * sizeof(double)));
    VG_HIP(hipMemcpyToSymbol(HIP_SYMBOL(cDiag), diag.data(), diag.size() * sizeof(double)));
    VG_HIP(hipMemcpyToSymbol(HIP_SYMBOL(cR1), r1.data(), r1.size() * sizeof(double)));
    VG_HIP(hipMemcpyToSymbol(HIP_SYMBOL(cR2), r2.data(), r2.size() * sizeof(double)));
    if (done.size() <= static_cast<size_t>(dev)) done.resize(static_cast<size_t>(dev) + 1, false);
    done[static_cast<size_t>(dev)] = true;
}

// The operator (and offset vector) indices that operators_build fills: the
// 16 M2M and L2L ones, then 16 + o for the 189 M2L offsets o of octant 0's
// walk.  A device table, written once per context.
void ops_selection(Ctx &c) {
    if (c.ops_sel.p) return;
    constexpr M2lSteps steps = m2l_steps();
    std::vector<int16_t> h(NOPS_USED);
    for (int i = 0; i < 16; ++i) h[static_cast<size_t>(i)] = static_cast<int16_t>(i);
    for (int i = 0; i < 189; ++i) h[static_cast<size_t>(16 + i)] = static_cast<int16_t>(16 + m2l_step(steps.d[i], steps.q[i], 0).o);
    c.ops_sel.ensure(NOPS_USED);
    VG_HIP(hipMemcpy(c.ops_sel.p, h.data(), NOPS_USED * sizeof(int16_t), hipMemcpyHostToDevice));
}

void operators_build(Ctx &c) {
    fmm_constants_init();
    // 8 M2M (child - parent), 8 L2L (parent - child) and 343 M2L (source -
    // target) offsets, formed on the device from the aspect ratio.  Only the
    // 189 M2L offsets of octant 0's walk are ever read (every octant uses them
    // through the mirror signs), so only those and the 16 M2M / L2L operators
    // are built; the other slots stay unwritten.
    const int nvec = 16 + 343;
    ops_selection(c);
    c.harm.ensure(static_cast<size_t>(nvec) * HSTRIDE);
    k_harmonics<<<NOPS_USED, 64, 0, c.stream>>>(c.ops_sel, nvec, c.box, 2 * c.p, c.harm);
    dim3 grid(NOPS_USED, ceil_div(c.K, OPS_ROWS));
    if (c.prec == 0) {
        c.op64.ensure(static_cast<size_t>(nvec) * c.K * c.K);
        k_ops<double><<<grid, 128 * OPS_ROWS, 0, c.stream>>>(c.ops_sel, c.harm, c.p, c.K, c.op64, nullptr);
    } else if (c.prec == 2) {
        c.op64.ensure(static_cast<size_t>(nvec) * c.K * c.K);
        k_ops<double><<<grid, 128 * OPS_ROWS, 0, c.stream>>>(c.ops_sel, c.harm, c.p, c.K, c.op64, nullptr);
        m2l_split_operators(c);
    } else {
        if (c.frag_K != c.K) {  // the padding, once for each order (the closure's fallback order may change)
            const size_t words = 343 * OpFrag(c.K).size(), words_ml = 16 * MlFrag(c.K).size();
            c.opfrag.ensure(words);
            c.op32.ensure(words_ml);
            VG_HIP(hipMemsetAsync(c.opfrag.p, 0, words * sizeof(float), c.stream));
            VG_HIP(hipMemsetAsync(c.op32.p, 0, words_ml * sizeof(float), c.stream));
            c.frag_K = c.K;
        }
        k_ops<float><<<grid, 128 * OPS_ROWS, 0, c.stream>>>(c.ops_sel, c.harm, c.p, c.K, c.op32, c.opfrag);
    }
    VG_LAUNCH_CHECK();
}

void fmm_upward(Ctx &c) {
    if (c.prec == 0)
        upward_t<double>(c);
    else
        upward_t<float>(c);
}

// Parts of the walked offsets of a grid of `grid` equal blocks: a CU's blocks
// share its matrix pipes, so the time goes with the fullest CU's share of the
// work, ceil(grid n / ncu) / n, and each part costs about 1 % (prologue, partial
// sums).  Grids of 8 and more blocks per CU are not cut.
int m2l_parts(unsigned grid, int ncu) {
    int best = 1;
    if (ncu <= 0 || grid >= 8u * static_cast<unsigned>(ncu)) return best;
    double t = 1e300;
    for (int n = 1; n <= 32; ++n) {
        const double x = static_cast<double>(ceil_div(static_cast<size_t>(grid) * n, ncu)) / n * (1 + 0.01 * n);
        if (x < t) t = x, best = n;
    }
    return best;
}

// Room for the partial sums of nsplit parts (nullptr for one), and their sum
// into the local expansions.
float *m2l_part_sums(Ctx &c, int np, int nsplit) {
    if (nsplit < 2) return nullptr;
    c.m2l_part.ensure(static_cast<size_t>(nsplit) * 8 * np * c.ldk * sizeof(float));
    return reinterpret_cast<float *>(c.m2l_part.p);
}
void m2l_add_parts(Ctx &c, const int32_t *parents, int np, int nsplit, const float *part) {
    if (nsplit < 2) return;
    k_m2l_sum<float><<<ceil_div(static_cast<size_t>(8) * np * c.K, 256), 256, 0, c.stream>>>(parents, np, c.t.child, c.t.count, nsplit, part, c.L32, c.K,
                                                                                          c.ldk);
    VG_LAUNCH_CHECK();
}

void fmm_m2l_plain_list(Ctx &c, const int32_t *parents, int np) {
    if (c.prec == 0)
        m2l_f64_list(c, parents, np);
    else
        m2l_f32_list(c, parents, np);
}

void fmm_m2l_plain(Ctx &c) {
    const TreeDev &t = c.t;
    // parents: internal cells of levels >= 1 (their children are the targets at level >= 2)
    if (t.depth < 1) return;
    const int64_t a = t.int_off[1], b = t.int_off.back();
    if (b > a) fmm_m2l_plain_list(c, t.int_ids.p + a, static_cast<int>(b - a));
}

void l2l_list(Ctx &c, const int32_t *parents, int64_t np) {
    if (np > 0) ml_level(c, parents, np, false);
    VG_LAUNCH_CHECK();
}

void l2p_flagged(Ctx &c, bool potential, const uint8_t *flag) { l2p_t<float>(c, potential, flag, true); }

void fmm_downward(Ctx &c, bool potential) {
    if (c.prec == 0)
        downward_t<double>(c, potential);
    else
        downward_t<float>(c, potential);
}

}  // namespace vg
