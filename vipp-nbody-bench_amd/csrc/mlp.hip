// mlp.hip - the learned closure's network: 28 -> 128 -> 128 -> 25, GELU on
// the hidden layers, FP16 weights and activations with FP32 accumulation in
// the forward pass (v_mfma_f32_16x16x16_f16), FP32 backward pass and Adam.
//
// Parameters are one FP32 vector (the master copy), row-major [out][in]:
//   W1 (128 x 28), b1 (128), W2 (128 x 128), b2 (128), W3 (25 x 128), b3 (25).
// The forward pass reads FP16 copies of W1..W3 prepacked in MFMA A-operand
// order; the backward pass uses the same FP16-rounded weights (as FP32), so
// the gradient is that of the function the forward pass evaluates (the FP16
// rounding of activations is passed straight through).
//
// Forward mapping: a wavefront evaluates 16 samples.  Layer l computes
// Z = W X^T: A = W (out x in, 16 x 16 tiles), B = X^T (in x samples).  For
// v_mfma_f32_16x16x16_f16, lane l holds A[l%16][4(l/16)+e], B[4(l/16)+e][l%16]
// and D[4(l/16)+r][l%16] (e, r = 0..3): the output tile t of one layer sits in
// the lanes exactly as the k-step t of the next layer's B operand, so hidden
// activations never leave registers.
#include "gravity.hpp"
#include "mlp.hpp"

#include <algorithm>
#include <cmath>
#include <numeric>
#include <random>

namespace vg {
namespace mlp {
namespace {

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

// A fragments: layer 1: 8 out-tiles x 2 k-steps, layer 2: 8 x 8, layer 3: 2 x 8
constexpr int F1 = 0, F2 = 16, F3 = 80, NFRAG = 96;
__host__ __device__ constexpr int frag_base(int layer) { return layer == 0 ? F1 : layer == 1 ? F2 : F3; }
__host__ __device__ constexpr int ksteps(int layer) { return layer == 0 ? 2 : 8; }

__device__ inline void gelu_factors(float z, float &f, float &g) { f = 0.5f * z, g = 1.0f + erff(z * 0.70710678118654752f); }
__device__ inline float gelu(float z) {
    float f, g;
    gelu_factors(z, f, g);
    return f * g;
}
__device__ inline float gelu_grad(float z) {
    return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// FP32 params -> FP16 A fragments [frag][lane][4] and FP16-rounded FP32 weights
__global__ __launch_bounds__(256) void k_pack(const float *__restrict__ par, _Float16 *__restrict__ frag, float *__restrict__ wr) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < NPAR) wr[i] = static_cast<float>(static_cast<_Float16>(par[i]));
    if (i >= NFRAG * 64) return;
    const int f = i / 64, l = i % 64;
    int layer, t, s;
    if (f < F2) layer = 0, t = f / 2, s = f % 2;
    else if (f < F3) layer = 1, t = (f - F2) / 8, s = (f - F2) % 8;
    else layer = 2, t = (f - F3) / 8, s = (f - F3) % 8;
    const int nin = layer == 0 ? IN : H, nout = layer == 2 ? OUT : H;
    const int woff = layer == 0 ? OW1 : layer == 1 ? OW2 : OW3;
    const int row = 16 * t + (l & 15);
    for (int e = 0; e < 4; ++e) {
        const int col = 16 * s + 4 * (l >> 4) + e;
        const float w = (row < nout && col < nin) ? par[woff + row * nin + col] : 0.0f;
        frag[(static_cast<int64_t>(f) * 64 + l) * 4 + e] = static_cast<_Float16>(w);
    }
}

// Forward pass of 16 samples per wavefront, 4 wavefronts per block.
__global__ __launch_bounds__(256) void k_forward(const half4 *__restrict__ frag, const float *__restrict__ par, const float *__restrict__ x, int64_t n,
                                                 float *__restrict__ y) {
    const int lane = threadIdx.x & 63;
    const int64_t j = (blockIdx.x * 4ll + (threadIdx.x >> 6)) * 16 + (lane & 15);  // this lane's sample
    const bool live = j < n;
    const int q = lane >> 4;                                                        // row group: rows 4q .. 4q+3 of a tile
    half4 b[8];
    // layer 1 input: k-step s holds inputs 16 s + 4 q + e
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = 16 * s + 4 * q + e;
            const float v = (live && k < IN) ? x[j * IN + k] : 0.0f;
            b[s][e] = static_cast<_Float16>(v);
        }
    half4 h[8];
#pragma unroll
    for (int layer = 0; layer < 2; ++layer) {
        const int ks = ksteps(layer);
        const float *bias = par + (layer == 0 ? OB1 : OB2);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            float4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < ks; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x16f16(frag[(frag_base(layer) + t * ks + s) * 64 + lane], b[s], acc, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int o = 16 * t + 4 * q + r;
                h[t][r] = static_cast<_Float16>(gelu(acc[r] + bias[o]));
            }
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) b[t] = h[t];
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        float4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 8; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x16f16(frag[(F3 + t * 8 + s) * 64 + lane], b[s], acc, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = 16 * t + 4 * q + r;
            if (live && o < OUT) y[j * OUT + o] = acc[r] + par[OB3 + o];
        }
    }
}

// f0 g0 and f1 g1, each rounded to FP16 once
__device__ inline uint32_t mul_f16x2(float f0, float g0, float f1, float g1) {
    uint32_t h = 0;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "+v"(h) : "v"(f0), "v"(g0));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(h) : "v"(f1), "v"(g1));
    return h;
}

// Forward and backward pass of 16 samples (rows idx[j] of x, t and w, or j
// itself without idx) by 8 wavefronts, up to what the weight gradients need: the
// FP16-rounded input (n x 32) and activations (n x 128), and
// dY = 2 w (y - t) / (W 25) with W the sum of the sample weights w (1 when
// none are given), dZ2 = (dY W3) * gelu'(Z2), dZ1 = (dZ2 W2) * gelu'(Z1).
// Also the block's weighted sum of squared errors.
//
// A batch of a few hundred samples is bound by latency: each wavefront takes one
// 16-output tile of a layer (hidden activations pass through LDS, in the order
// k_forward's registers have) and, on the way back, one column of four samples,
// so that a weight is read once for the four.  16 us for 512 samples; fragments
// or weights loaded ahead of their use were slower (22 us, or spilled).
__global__ __launch_bounds__(512) void k_train(const half4 *__restrict__ frag, const float *__restrict__ par, const float *__restrict__ wr,
                                               const float *__restrict__ x, const float *__restrict__ tgt, const float *__restrict__ wt,
                                               const uint32_t *__restrict__ idx, int64_t n, float inv_count, float *__restrict__ x16,
                                               float *__restrict__ a1, float *__restrict__ a2, float *__restrict__ dy, float *__restrict__ dz1,
                                               float *__restrict__ dz2, float *__restrict__ sse) {
    constexpr int LZ = H + 4;  // floats between samples in LDS
    __shared__ half4 s_h[2][8][64];
    __shared__ float s_z[2][16 * LZ];
    __shared__ float s_dy[16 * 28], s_dz2[16 * LZ], s_err[2];
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, u = lane & 15;
    const int t = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t j0 = blockIdx.x * 16ll, j = j0 + u;  // forward: this lane's sample
    const bool live = j < n;
    const int64_t row = !live ? 0 : idx ? idx[j] : j;
    half4 b[8];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = 16 * s + 4 * q + e;
            b[s][e] = static_cast<_Float16>((live && k < IN) ? x[row * IN + k] : 0.0f);
        }
        if (t == 0 && live)
            *reinterpret_cast<float4v *>(x16 + j * 32 + 16 * s + 4 * q) = float4v{static_cast<float>(b[s][0]), static_cast<float>(b[s][1]),
                                                                                  static_cast<float>(b[s][2]), static_cast<float>(b[s][3])};
    }
#pragma unroll
    for (int layer = 0; layer < 2; ++layer) {
        const int ks = ksteps(layer);
        float4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < ks; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x16f16(frag[(frag_base(layer) + t * ks + s) * 64 + lane], b[s], acc, 0, 0, 0);
        const int o = 16 * t + 4 * q;
        const float *bias = par + (layer == 0 ? OB1 : OB2) + o;
        float4v z, a;
        float f[4], g[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            z[r] = acc[r] + bias[r];
            gelu_factors(z[r], f[r], g[r]);
        }
        const half4 h = __builtin_bit_cast(half4, make_uint2(mul_f16x2(f[0], g[0], f[1], g[1]), mul_f16x2(f[2], g[2], f[3], g[3])));
#pragma unroll
        for (int r = 0; r < 4; ++r) a[r] = static_cast<float>(h[r]);
        *reinterpret_cast<float4v *>(&s_z[layer][u * LZ + o]) = z;
        s_h[layer][t][lane] = h;
        if (live) *reinterpret_cast<float4v *>((layer == 0 ? a1 : a2) + j * H + o) = a;
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 8; ++s) b[s] = s_h[layer][s][lane];
    }
    if (t < 2) {
        float4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 8; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x16f16(frag[(F3 + t * 8 + s) * 64 + lane], b[s], acc, 0, 0, 0);
        const float wj = live && wt ? wt[row] : 1.0f;
        float err = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = 16 * t + 4 * q + r;
            if (o >= 28) continue;
            float g = 0.0f;
            if (live && o < OUT) {
                const float d = acc[r] + par[OB3 + o] - tgt[row * OUT + o];
                err += wj * d * d;
                g = 2.0f * wj * d * inv_count;
                dy[j * OUT + o] = g;
            }
            s_dy[u * 28 + o] = g;
        }
        for (int w = 32; w > 0; w >>= 1) err += __shfl_xor(err, w);
        if (lane == 0) s_err[t] = err;
    }
    __syncthreads();
    if (tid == 0) sse[blockIdx.x] = s_err[0] + s_err[1];
    const int h = tid & 127, u0 = (tid >> 7) * 4;  // backward: this thread's column and samples
    float g[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int o = 0; o < OUT; ++o) {
        const float w = wr[OW3 + o * H + h];
#pragma unroll
        for (int e = 0; e < 4; ++e) g[e] += s_dy[(u0 + e) * 28 + o] * w;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float d2 = g[e] * gelu_grad(s_z[1][(u0 + e) * LZ + h]);
        s_dz2[(u0 + e) * LZ + h] = d2;
        if (j0 + u0 + e < n) dz2[(j0 + u0 + e) * H + h] = d2;
        g[e] = 0.0f;
    }
    __syncthreads();
#pragma unroll 4
    for (int o = 0; o < H; o += 4) {
        float w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = wr[OW2 + (o + k) * H + h];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float4v d = *reinterpret_cast<const float4v *>(&s_dz2[(u0 + e) * LZ + o]);
#pragma unroll
            for (int k = 0; k < 4; ++k) g[e] += d[k] * w[k];
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (j0 + u0 + e < n) dz1[(j0 + u0 + e) * H + h] = g[e] * gelu_grad(s_z[0][(u0 + e) * LZ + h]);
}

struct AdamStep {
    float lr, b1, b2, eps, c1, c2;
};

// Weight gradients of the three layers, dW[o][i] = sum_j dZ[j][o] A[j][i] and
// db[o] = sum_j dZ[j][o] (a column of ones beside A), each sum by one thread in the
// order of the samples (deterministic); with ADAM the thread then takes the
// parameter's step, its FP16 copies included, otherwise the gradient is stored.
//
// A block takes 4 outputs (one per wavefront) by 64 columns of one layer: 149
// blocks, so that the serial sums spread over the chip; 128 samples at a time
// come through LDS, the next 128 on their way meanwhile (256 were slower: 13 ->
// 18 us).  512 samples: 3 x 126 us with one thread per weight reading its terms
// from memory one by one -> 13 us; an epoch of 20,000 samples in batches of
// 512: 20.3 -> 1.7 ms, of which 1.2 are kernels and the rest copies and buffers.
constexpr int WG_SAMPLES = 128, WG1 = H / 4, WG2 = H / 4 * 3, WG3 = (OUT + 3) / 4 * 3;
template <bool ADAM>
__global__ __launch_bounds__(256) void k_weights(const float *__restrict__ x16, const float *__restrict__ a1, const float *__restrict__ a2,
                                                 const float *__restrict__ dz1, const float *__restrict__ dz2, const float *__restrict__ dy, int64_t n,
                                                 float *__restrict__ grad, AdamStep st, float *__restrict__ par, float *__restrict__ m,
                                                 float *__restrict__ v, float *__restrict__ wr, _Float16 *__restrict__ frag) {
    __shared__ float s_a[WG_SAMPLES][64];
    __shared__ float4v s_d[4][WG_SAMPLES / 4];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    int blk = blockIdx.x, layer = 0;
    if (blk >= WG1) blk -= WG1, layer = 1;
    if (layer == 1 && blk >= WG2) blk -= WG2, layer = 2;
    const int nin = layer == 0 ? IN : H, nout = layer == 2 ? OUT : H, lda = layer == 0 ? 32 : H, nc = layer == 0 ? 1 : 3;
    const float *A = layer == 0 ? x16 : layer == 1 ? a1 : a2, *D = layer == 0 ? dz1 : layer == 1 ? dz2 : dy;
    const int o0 = blk / nc * 4, col = blk % nc * 64 + lane, o = o0 + wv;
    constexpr int NA = WG_SAMPLES / 4, ND = WG_SAMPLES / 64;  // words a thread brings
    float va[NA], vd[ND];
    auto fetch = [&](int64_t b) {
#pragma unroll
        for (int k = 0; k < NA; ++k) {
            const int64_t j = b + 4 * k + wv;
            va[k] = j < n && col < nin ? A[j * lda + col] : col == nin ? 1.0f : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            const int64_t j = b + 64 * k + (tid >> 2);
            const int od = o0 + (tid & 3);
            vd[k] = j < n && od < nout ? D[j * nout + od] : 0.0f;
        }
    };
    fetch(0);
    float s = 0.0f;
    for (int64_t b = 0; b < n; b += WG_SAMPLES) {
#pragma unroll
        for (int k = 0; k < NA; ++k) s_a[4 * k + wv][lane] = va[k];
#pragma unroll
        for (int k = 0; k < ND; ++k) reinterpret_cast<float *>(s_d[tid & 3])[64 * k + (tid >> 2)] = vd[k];
        __syncthreads();
        if (b + WG_SAMPLES < n) fetch(b + WG_SAMPLES);
#pragma unroll 8
        for (int k = 0; k < WG_SAMPLES / 4; ++k) {
            const float4v d = s_d[wv][k];
#pragma unroll
            for (int e = 0; e < 4; ++e) s += d[e] * s_a[4 * k + e][lane];
        }
        __syncthreads();
    }
    if (o >= nout || col > nin) return;
    const bool bias = col == nin;
    const int i = bias ? (layer == 0 ? OB1 : layer == 1 ? OB2 : OB3) + o : (layer == 0 ? OW1 : layer == 1 ? OW2 : OW3) + o * nin + col;
    if (!ADAM) {
        grad[i] = s;
        return;
    }
    const float mi = st.b1 * m[i] + (1.0f - st.b1) * s;
    const float vi = st.b2 * v[i] + (1.0f - st.b2) * s * s;
    m[i] = mi;
    v[i] = vi;
    const float w = par[i] - st.lr * (mi / st.c1) / (sqrtf(vi / st.c2) + st.eps);
    par[i] = w;
    const _Float16 wh = static_cast<_Float16>(w);
    wr[i] = static_cast<float>(wh);
    if (!bias)  // its place in the A fragments (k_pack)
        frag[((frag_base(layer) + (o >> 4) * ksteps(layer) + (col >> 4)) * 64 + (o & 15) + 16 * (col >> 2 & 3)) * 4 + (col & 3)] = wh;
}

}  // namespace

void Net::set_params(hipStream_t st, const float *par_dev) {
    frag.ensure(NFRAG * 64 * 4);
    wr.ensure(NPAR);
    if (par_dev != par.p) {
        par.ensure(NPAR);
        VG_HIP(hipMemcpyAsync(par.p, par_dev, NPAR * sizeof(float), hipMemcpyDeviceToDevice, st));
    }
    k_pack<<<ceil_div(std::max(NPAR, NFRAG * 64), 256), 256, 0, st>>>(par, frag, wr);
    VG_LAUNCH_CHECK();
}

void Net::forward(hipStream_t st, const float *x, int64_t n, float *y) const {
    if (n <= 0) return;
    k_forward<<<ceil_div(n, 64), 256, 0, st>>>(reinterpret_cast<const half4 *>(frag.p), par, x, n, y);
    VG_LAUNCH_CHECK();
}

int64_t Net::loss_terms(int64_t n) { return ceil_div(n, 16); }

void Net::activations(hipStream_t st, const float *x, const float *t, const float *w, const uint32_t *idx, double wsum, int64_t n, float *sse) {
    x16.ensure(n * 32);
    a1.ensure(n * H), a2.ensure(n * H);
    dy.ensure(n * OUT), dz1.ensure(n * H), dz2.ensure(n * H);
    k_train<<<static_cast<unsigned>(loss_terms(n)), 512, 0, st>>>(reinterpret_cast<const half4 *>(frag.p), par, wr, x, t, w, idx, n,
                                                                  static_cast<float>(1.0 / (wsum * OUT)), x16, a1, a2, dy, dz1, dz2, sse);
    VG_LAUNCH_CHECK();
}

float Net::loss_grad(hipStream_t st, const float *x, const float *t, const float *w, double wsum, int64_t n, float *grad) {
    DevBuf<float> sse;
    std::vector<float> h(static_cast<size_t>(loss_terms(n)));
    sse.ensure(h.size());
    const double wtot = w ? wsum : static_cast<double>(n);
    activations(st, x, t, w, nullptr, wtot, n, sse);
    k_weights<false><<<WG1 + WG2 + WG3, 256, 0, st>>>(x16, a1, a2, dz1, dz2, dy, n, grad, AdamStep{}, nullptr, nullptr, nullptr, nullptr, nullptr);
    VG_LAUNCH_CHECK();
    VG_HIP(hipMemcpyAsync(h.data(), sse.p, h.size() * sizeof(float), hipMemcpyDeviceToHost, st));
    VG_HIP(hipStreamSynchronize(st));
    double s = 0;
    for (float e : h) s += e;
    return static_cast<float>(s / (wtot * OUT));
}

void Net::train_step(hipStream_t st, const float *x, const float *t, const float *w, const uint32_t *idx, double wsum, int64_t n, float lr, int step,
                     float *sse) {
    if (m.cap < static_cast<size_t>(NPAR)) {
        m.ensure(NPAR), v.ensure(NPAR);
        VG_HIP(hipMemsetAsync(m.p, 0, NPAR * sizeof(float), st));
        VG_HIP(hipMemsetAsync(v.p, 0, NPAR * sizeof(float), st));
    }
    activations(st, x, t, w, idx, wsum, n, sse);
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - std::pow(b1, static_cast<float>(step)), c2 = 1.0f - std::pow(b2, static_cast<float>(step));
    k_weights<true><<<WG1 + WG2 + WG3, 256, 0, st>>>(x16, a1, a2, dz1, dz2, dy, n, nullptr, AdamStep{lr, b1, b2, 1e-8f, c1, c2}, par, m, v, wr, frag);
    VG_LAUNCH_CHECK();
}

}  // namespace mlp
}  // namespace vg
