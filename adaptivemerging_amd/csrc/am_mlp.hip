// am_mlp.hip - learned warm start: per-contact features, a 24-64-64-64-3 ReLU
// MLP with BF16 weights on the CDNA matrix cores (v_mfma_f32_16x16x16_bf16,
// FP32 accumulation), its backward pass and an Adam update, and the
// start-quality residual that decides between the learned and the plain start.
//
// Feature vector (24 FP32, dimensionless), per contact with solve bodies a, b:
//   0-2 normal, 3-5 tangent 1 (world; tangent 2 = n x t1 adds nothing),
//   6 1 when the plain warm start found no previous contact (new this step),
//   7-8 0,
//   9-11 constraint-space velocity J (v_a, w_a, v_b, w_b) / (g dt),
//   12 violation / (g dt^2),
//   13 minv_a / (minv_a + minv_b), 14 log10((minv_a + minv_b) * 1 kg) / 3,
//   15-17 diag(jinv_a) / trace(jinv_a), 18-20 same for b (0 when pinned),
//   21-23 slog(previous-frame lambda / S),
// with S = g dt / D_nn (D_nn = J_n M^-1 J_n^T) and slog(x) = sign(x) ln(1 + |x|),
// which keeps the impulses of a 100:1 mass-ratio pile in a range BF16 holds.
// The network predicts the change of slog(lambda / S) from the plain start,
// bounded by kMaxLogStep.
#include "am_mlp.hpp"

namespace am {

typedef short short4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// features
AMD_INLINE double slog(double x) { return x < 0 ? -log1p(-x) : log1p(x); }
AMD_INLINE double sexp(double z) { return z < 0 ? -expm1(-z) : expm1(z); }
constexpr double kMaxLogStep = 2.0;  // largest change of slog(lambda / S) a prediction makes

__global__ void k_features(FeatureArgs F) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= F.n) return;
    const BodiesView& B = F.B;
    const ContactsView& C = F.C;
    int b1 = C.b1[k], b2 = C.b2[k];
    int a = B.parent[b1] >= 0 ? B.parent[b1] : b1;
    int b = B.parent[b2] >= 0 ? B.parent[b2] : b2;
    const double* J = &C.J[(size_t)k * 36];
    float* f = &F.out[(size_t)k * kMlpIn];
    double gdt = F.g * F.dt;
    // frame (jb.v of the normal and first tangent rows)
    for (int r = 0; r < 2; r++)
        for (int i = 0; i < 3; i++) f[r * 3 + i] = (float)J[r * 12 + 6 + i];
    f[6] = C.is_new[k] ? 1.f : 0.f;
    f[7] = 0.f;
    f[8] = 0.f;
    d3 va = ld3(&B.v[a * 3]), wa = ld3(&B.w[a * 3]), vb = ld3(&B.v[b * 3]), wb = ld3(&B.w[b * 3]);
    for (int r = 0; r < 3; r++) {
        const double* row = J + r * 12;
        double u = dot(ld3(row), va) + dot(ld3(row + 3), wa) + dot(ld3(row + 6), vb) + dot(ld3(row + 9), wb);
        f[9 + r] = (float)(u / gdt);
    }
    f[12] = (float)(C.viol[k] / (gdt * F.dt));
    double ma = B.minv[a], mb = B.minv[b];
    double msum = ma + mb;
    f[13] = (float)(msum > 0 ? ma / msum : 0.5);
    f[14] = (float)(log10(msum + 1e-12) / 3.0);
    const int ids[2] = {a, b};
    for (int s = 0; s < 2; s++) {
        const double* Ji = &B.jinv[ids[s] * 9];
        double tr = Ji[0] + Ji[4] + Ji[8];
        for (int i = 0; i < 3; i++) f[15 + s * 3 + i] = (float)(tr > 0 ? Ji[i * 4] / tr : 0.0);
    }
    // D_nn (Contact.computeJMinvJt normal row)
    d3 t1 = mul(ldm(&B.jinv[a * 9]), ld3(J + 3));
    d3 t2 = mul(ldm(&B.jinv[b * 9]), ld3(J + 9));
    double D = ma * dot(ld3(J), ld3(J)) + dot(ld3(J + 3), t1) + mb * dot(ld3(J + 6), ld3(J + 6)) + dot(ld3(J + 9), t2);
    double S = D > 0 ? gdt / D : 1.0;
    F.scale[k] = S;
    for (int r = 0; r < 3; r++) f[21 + r] = (float)slog(C.lam[k * 3 + r] / S);
}

void launch_features(hipStream_t s, const FeatureArgs& F) {
    if (F.n > 0) hipLaunchKernelGGL(k_features, dim3((F.n + 127) / 128), dim3(128), 0, s, F);
}

// ---------------------------------------------------------------------------
// BF16 helpers (round to nearest even)
AMD_INLINE unsigned short f2bf(float f) {
    unsigned u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)(u >> 16);  // inf / nan
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}
AMD_INLINE float bf2f(unsigned short h) { return __uint_as_float(((unsigned)h) << 16); }

// Layer geometry: padded input 32, hidden 64, padded output 16.
constexpr int kIn = 32, kH = 64, kOut = 16;

// Every product runs transposed, D (n x rows) = W^T (n x k) * in^T (k x rows),
// on v_mfma_f32_16x16x16_bf16: lane l holds A[l%16][4(l/16)+j],
// B[4(l/16)+j][l%16] and D[4(l/16)+j][l%16] for j = 0..3.  With the weights
// stored [out][in] and the activations [row][unit], each lane's four operand
// values are one 8-byte LDS read, and its four results are consecutive units
// of one row, one 8-byte write of the next layer's input.  Rows are padded by
// 8 values so that the 16 lanes of a fragment start on different banks.
constexpr int kInS = kIn + 8, kHS = kH + 8, kOutS = kOut + 4;
typedef short4v __attribute__((may_alias)) short4a;
AMD_INLINE short4v ld4(const unsigned short* p) { return *reinterpret_cast<const short4a*>(p); }
AMD_INLINE void st4(unsigned short* p, const unsigned short (&v)[4]) {
    short4v s = {(short)v[0], (short)v[1], (short)v[2], (short)v[3]};
    *reinterpret_cast<short4a*>(p) = s;
}
AMD_INLINE float4v mfma16(short4v a, short4v b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
// LDS of one wave is read back by other lanes of it: order the accesses.
AMD_INLINE void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Weights in LDS as [out][in] (forward), biases.
struct MlpLds {
    alignas(16) unsigned short t1[kH * kInS];
    alignas(16) unsigned short t2[kH * kHS];
    alignas(16) unsigned short t3[kH * kHS];
    alignas(16) unsigned short t4[kOut * kHS];
    float b1[kH], b2[kH], b3[kH], b4[kOut];
};
// The same weights as [in][out], which the backward pass multiplies by.
struct MlpLdsBack {
    alignas(16) unsigned short w2[kH * kHS];
    alignas(16) unsigned short w3[kH * kHS];
    alignas(16) unsigned short w4[kH * kOutS];
};

// one matrix of `in` rows and `out` (16 or 64) columns, four values a thread
AMD_INLINE void load_matrix(const unsigned short* W, int in, int out, unsigned short* t, int ts, unsigned short* w,
                            int ws) {
    for (int i = threadIdx.x; i < in * out / 4; i += blockDim.x) {
        const int r = i / (out / 4), c = (i % (out / 4)) * 4;
        const short4v v = ld4(W + r * out + c);
#pragma unroll
        for (int j = 0; j < 4; j++) t[(c + j) * ts + r] = (unsigned short)v[j];
        if (w) *reinterpret_cast<short4a*>(w + r * ws + c) = v;
    }
}
AMD_INLINE void load_weights(const MlpWeights& W, MlpLds& L, MlpLdsBack* B) {
    load_matrix(W.w1_bf, kIn, kH, L.t1, kInS, nullptr, 0);
    load_matrix(W.w2_bf, kH, kH, L.t2, kHS, B ? B->w2 : nullptr, kHS);
    load_matrix(W.w3_bf, kH, kH, L.t3, kHS, B ? B->w3 : nullptr, kHS);
    load_matrix(W.w4_bf, kH, kOut, L.t4, kHS, B ? B->w4 : nullptr, kOutS);
    for (int i = threadIdx.x; i < kH; i += blockDim.x) {
        L.b1[i] = W.b1[i];
        L.b2[i] = W.b2[i];
        L.b3[i] = W.b3[i];
    }
    for (int i = threadIdx.x; i < kOut; i += blockDim.x) L.b4[i] = W.b4[i];
    __syncthreads();
}

// Activations of one wave's 16-row tile, bf16: the input and two layers in
// turn as [row][unit]; for the backward pass also every layer as [unit][row]
// (the operands of the weights' gradients, whose sums run over rows).
struct WaveAct {
    alignas(16) unsigned short x[16 * kInS];
    alignas(16) unsigned short h[2][16 * kHS];
};
struct WaveBack {
    alignas(16) unsigned short xt[kIn * 16];
    alignas(16) unsigned short ht[3][kH * 16];
    alignas(16) unsigned short dy[16 * kOutS];
    alignas(16) unsigned short dyt[kOut * 16];
    alignas(16) unsigned short dt[kH * 16];
};

constexpr int kMlpWaves = 4;

// out (16 x 64) = relu(in (16 x K) W + bias); with outt also as [unit][row],
// and with mask bit 4 t + j set where this lane's unit 16 t + 4 (l/16) + j is positive
template <int K>
AMD_INLINE void dense_relu(const unsigned short* wt, int ws, const unsigned short* in, int is, const float* bias,
                           unsigned short* out, unsigned short* outt, unsigned* mask) {
    const int col = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
    short4v b[K / 16];
#pragma unroll
    for (int k = 0; k < K / 16; k++) b[k] = ld4(in + col * is + k * 16 + 4 * q);
    unsigned m = 0;
#pragma unroll
    for (int t = 0; t < kH / 16; t++) {
        float4v c = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < K / 16; k++) c = mfma16(ld4(wt + (t * 16 + col) * ws + k * 16 + 4 * q), b[k], c);
        unsigned short v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float z = c[j] + bias[t * 16 + 4 * q + j];
            v[j] = f2bf(z > 0.f ? z : 0.f);
            if (outt) outt[(t * 16 + 4 * q + j) * 16 + col] = v[j];
            m |= (v[j] != 0 ? 1u : 0u) << (4 * t + j);
        }
        st4(out + col * kHS + t * 16 + 4 * q, v);
    }
    if (mask) *mask = m;
}

// A tile's input rows (24 floats each, row r of X at rows(r); a missing row
// and the padding columns read 0): four lanes a row, six floats each.
template <class F>
AMD_INLINE void load_x_tile(const float* X, int row0, int n, F rows, unsigned short* x, unsigned short* xt) {
    const int l = threadIdx.x & 63, r = l >> 2, c0 = 6 * (l & 3);
    float v[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (row0 + r < n) {
        const float2* src = reinterpret_cast<const float2*>(X + (size_t)rows(row0 + r) * kMlpIn + c0);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const float2 p = src[i];
            v[2 * i] = p.x;
            v[2 * i + 1] = p.y;
        }
    }
#pragma unroll
    for (int i = 0; i < 6; i++) {
        const unsigned short h = f2bf(v[i]);
        x[r * kInS + c0 + i] = h;
        if (xt) xt[(c0 + i) * 16 + r] = h;
    }
}
AMD_INLINE void clear_x_padding(unsigned short* x, unsigned short* xt) {
    const int l = threadIdx.x & 63;
    for (int i = l; i < 16 * (kIn - kMlpIn); i += 64) {
        x[(i & 15) * kInS + kMlpIn + (i >> 4)] = 0;
        if (xt) xt[kMlpIn * 16 + i] = 0;
    }
}
// the output layer: lane l holds unit 4 (l/16) + j of row l%16
AMD_INLINE float4v out_layer(const MlpLds& L, const unsigned short* h) {
    const int col = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
    float4v c = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < kH / 16; k++)
        c = mfma16(ld4(L.t4 + col * kHS + k * 16 + 4 * q), ld4(h + col * kHS + k * 16 + 4 * q), c);
    return c;
}

// forward: Y[n x 3] = mlp(X[n x 24])
__global__ __launch_bounds__(kMlpWaves * 64) void k_mlp_forward(MlpWeights W, const float* X, int n, float* Y) {
    __shared__ MlpLds L;
    __shared__ WaveAct act[kMlpWaves];
    load_weights(W, L, nullptr);
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
    WaveAct& A = act[wave];
    clear_x_padding(A.x, nullptr);
    const int tiles = (n + 15) / 16;
    for (int tile = blockIdx.x * kMlpWaves + wave; tile < tiles; tile += gridDim.x * kMlpWaves) {
        const int row0 = tile * 16;
        load_x_tile(X, row0, n, [](int r) { return r; }, A.x, nullptr);
        wave_sync();
        dense_relu<kIn>(L.t1, kInS, A.x, kInS, L.b1, A.h[0], nullptr, nullptr);
        wave_sync();
        dense_relu<kH>(L.t2, kHS, A.h[0], kHS, L.b2, A.h[1], nullptr, nullptr);
        wave_sync();
        dense_relu<kH>(L.t3, kHS, A.h[1], kHS, L.b3, A.h[0], nullptr, nullptr);
        wave_sync();
        const float4v c = out_layer(L, A.h[0]);
        const int row = row0 + (l & 15);
        if (l < 16 && row < n)
#pragma unroll
            for (int j = 0; j < kMlpOut; j++) Y[(size_t)row * kMlpOut + j] = c[j] + L.b4[j];
        wave_sync();
    }
}

void launch_mlp_forward(hipStream_t s, const MlpWeights& W, const float* X, int n, float* Y) {
    if (n <= 0) return;
    int tiles = (n + 15) / 16;
    int blocks = std::min((tiles + kMlpWaves - 1) / kMlpWaves, 1024);
    hipLaunchKernelGGL(k_mlp_forward, dim3(blocks), dim3(kMlpWaves * 64), 0, s, W, X, n, Y);
}

// ---------------------------------------------------------------------------
// backward: loss = sum over rows of |y - t|^2 / n_total, rows = idx[0..n) of
// X/T (all in order when idx is null).
//
// Each wave keeps the gradients of every weight in matrix accumulators over
// all its tiles (44 of 16 x 16, 176 registers: one workgroup a CU gives a wave
// 512) and writes them once, to its own part of `partial`; k_grad_apply sums
// the parts.  Bound by latency: the chain of layers of a tile, and at a batch
// of 256 the copy of the weights into LDS.  Measured: 42 us for 20,001 rows
// and 22 us for a batch of 256, the sums 11 and 5 us more.  A form that added
// each tile's gradients to the weights with atomics spent its time on those
// (2636 and 80 us).

// dh (16 x 64) = (dnext (16 x KN) W^T) * relu'(h): w is [64][KN] with stride
// ws, dnext [row][KN]; written as [row][unit] (when dh is not null) and
// [unit][row]; unrounded column sums go to db.
template <int KN>
AMD_INLINE void back_layer(const unsigned short* w, int ws, const unsigned short* dnext, int ds, unsigned mask,
                           bool valid, unsigned short* dh, unsigned short* dt, float4v (&db)[kH / 16]) {
    const int col = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
    short4v b[KN / 16];
#pragma unroll
    for (int k = 0; k < KN / 16; k++) b[k] = ld4(dnext + col * ds + k * 16 + 4 * q);
#pragma unroll
    for (int t = 0; t < kH / 16; t++) {
        float4v c = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < KN / 16; k++) c = mfma16(ld4(w + (t * 16 + col) * ws + k * 16 + 4 * q), b[k], c);
        unsigned short v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float g = valid && ((mask >> (4 * t + j)) & 1u) ? c[j] : 0.f;
            db[t][j] += g;
            v[j] = f2bf(g);
            dt[(t * 16 + 4 * q + j) * 16 + col] = v[j];
        }
        if (dh) st4(dh + col * kHS + t * 16 + 4 * q, v);
    }
}
// dW (16 M x 64) += in^T dh over the tile's 16 rows, both as [unit][row]
template <int M>
AMD_INLINE void weight_grad(const unsigned short* int_, const unsigned short* dt, float4v (&g)[M][kH / 16]) {
    const int col = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
    short4v b[kH / 16];
#pragma unroll
    for (int t = 0; t < kH / 16; t++) b[t] = ld4(dt + (t * 16 + col) * 16 + 4 * q);
#pragma unroll
    for (int m = 0; m < M; m++) {
        const short4v a = ld4(int_ + (m * 16 + col) * 16 + 4 * q);
#pragma unroll
        for (int t = 0; t < kH / 16; t++) g[m][t] = mfma16(a, b[t], g[m][t]);
    }
}
template <int M>
AMD_INLINE void store_grad(const float4v (&g)[M][kH / 16], float* out) {
    const int col = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int t = 0; t < kH / 16; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) out[(m * 16 + 4 * q + j) * kH + t * 16 + col] = g[m][t][j];
}
// sum over the 16 rows (lanes l % 16) of each of the lane's units
AMD_INLINE void store_bias(const float4v (&db)[kH / 16], float* out) {
    const int col = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int t = 0; t < kH / 16; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float v = db[t][j];
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o, 64);
            if (col == 0) out[t * 16 + 4 * q + j] = v;
        }
}

__global__ __launch_bounds__(kMlpWaves * 64) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_mlp_backward(
    MlpWeights W, const float* X, const float* T, const int* idx, int n, float inv_total, float* partial) {
    __shared__ MlpLds L;
    __shared__ MlpLdsBack LB;
    __shared__ WaveAct act[kMlpWaves];
    __shared__ WaveBack back[kMlpWaves];
    load_weights(W, L, &LB);
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, col = l & 15, q = l >> 4;
    WaveAct& A = act[wave];
    WaveBack& K = back[wave];
    clear_x_padding(A.x, K.xt);
    const int tiles = (n + 15) / 16;
    auto source = [&](int r) { return idx ? idx[r] : r; };
    const float4v zero = {0, 0, 0, 0};
    float4v g1[kIn / 16][kH / 16], g2[kH / 16][kH / 16], g3[kH / 16][kH / 16], g4[kH / 16];
    float4v s1[kH / 16], s2[kH / 16], s3[kH / 16], s4 = zero;
#pragma unroll
    for (int t = 0; t < kH / 16; t++) {
#pragma unroll
        for (int m = 0; m < kH / 16; m++) {
            if (m < kIn / 16) g1[m][t] = zero;
            g2[m][t] = zero;
            g3[m][t] = zero;
        }
        g4[t] = s1[t] = s2[t] = s3[t] = zero;
    }
    float my_loss = 0.f;
    for (int tile = blockIdx.x * kMlpWaves + wave; tile < tiles; tile += gridDim.x * kMlpWaves) {
        const int row0 = tile * 16;
        const bool valid = row0 + col < n;
        unsigned m1, m2, m3;
        load_x_tile(X, row0, n, source, A.x, K.xt);
        wave_sync();
        dense_relu<kIn>(L.t1, kInS, A.x, kInS, L.b1, A.h[0], K.ht[0], &m1);
        wave_sync();
        dense_relu<kH>(L.t2, kHS, A.h[0], kHS, L.b2, A.h[1], K.ht[1], &m2);
        wave_sync();
        dense_relu<kH>(L.t3, kHS, A.h[1], kHS, L.b3, A.h[0], K.ht[2], &m3);
        wave_sync();
        // output layer and dL/dy = 2 (y - t) / n_total: units 0-2 sit in lanes 0-15
        const float4v c = out_layer(L, A.h[0]);
        unsigned short d[4] = {0, 0, 0, 0};
        if (q == 0 && valid) {
            const float* want = T + (size_t)source(row0 + col) * kMlpOut;
#pragma unroll
            for (int j = 0; j < kMlpOut; j++) {
                const float e = c[j] + L.b4[j] - want[j];
                my_loss += e * e * inv_total;
                const float g = 2.f * e * inv_total;
                s4[j] += g;
                d[j] = f2bf(g);
            }
        }
        st4(K.dy + col * kOutS + 4 * q, d);
#pragma unroll
        for (int j = 0; j < 4; j++) K.dyt[(4 * q + j) * 16 + col] = d[j];
        wave_sync();
        // dW4 (64 x 16) += h3^T dy
        {
            const short4v b = ld4(K.dyt + col * 16 + 4 * q);
#pragma unroll
            for (int m = 0; m < kH / 16; m++) g4[m] = mfma16(ld4(K.ht[2] + (m * 16 + col) * 16 + 4 * q), b, g4[m]);
        }
        // back through layers 3, 2, 1
        back_layer<kOut>(LB.w4, kOutS, K.dy, kOutS, m3, valid, A.h[1], K.dt, s3);
        wave_sync();
        weight_grad<kH / 16>(K.ht[1], K.dt, g3);
        wave_sync();
        back_layer<kH>(LB.w3, kHS, A.h[1], kHS, m2, valid, A.h[0], K.dt, s2);
        wave_sync();
        weight_grad<kH / 16>(K.ht[0], K.dt, g2);
        wave_sync();
        back_layer<kH>(LB.w2, kHS, A.h[0], kHS, m1, valid, nullptr, K.dt, s1);
        wave_sync();
        weight_grad<kIn / 16>(K.xt, K.dt, g1);
        wave_sync();
    }
    float* out = partial + (size_t)(blockIdx.x * kMlpWaves + wave) * kPartial;
    store_grad(g1, out);
    out += kPadW1;
    store_grad(g2, out);
    out += kPadW2;
    store_grad(g3, out);
    out += kPadW3;
#pragma unroll
    for (int m = 0; m < kH / 16; m++)
#pragma unroll
        for (int j = 0; j < 4; j++) out[(m * 16 + 4 * q + j) * kOut + col] = g4[m][j];
    out += kPadW4;
    store_bias(s1, out);
    store_bias(s2, out + kPadB1);
    store_bias(s3, out + kPadB1 + kPadB2);
    out += kPadB1 + kPadB2 + kPadB3;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float v = s4[j];
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o, 64);
        if (col == 0) out[4 * q + j] = v;
    }
    for (int o = 32; o > 0; o >>= 1) my_loss += __shfl_xor(my_loss, o, 64);
    if (l == 0) out[kPadB4] = my_loss;
}

// Sums the waves' partial gradients in a fixed order, 64 parameters a
// workgroup, 16 threads each (a thread alone would walk the parts of all the
// waves one load after the other); then, with P.p set, the Adam update of the
// FP32 master weights and their BF16 copies, else the sums go to P.g.  The
// last entry is the loss, added to *loss.
__global__ __launch_bounds__(1024) void k_grad_apply(AdamArgs P, const float* partial, int parts, float* loss) {
    __shared__ float sum[16][64];
    const int e = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + e;
    float g = 0.f;
    if (i <= kPadTotal)
        for (int k = w; k < parts; k += 16) g += partial[(size_t)k * kPartial + i];
    sum[w][e] = g;
    __syncthreads();
    if (w != 0 || i > kPadTotal) return;
#pragma unroll
    for (int k = 1; k < 16; k++) g += sum[k][e];
    if (i == kPadTotal) {
        *loss += g;
        return;
    }
    if (!P.p) {
        P.g[i] = g;
        return;
    }
    float mi = P.b1 * P.m[i] + (1.f - P.b1) * g;
    float vi = P.b2 * P.v[i] + (1.f - P.b2) * g * g;
    P.m[i] = mi;
    P.v[i] = vi;
    float pi = P.p[i] - P.lr * (mi / P.c1) / (sqrtf(vi / P.c2) + P.eps);
    P.p[i] = pi;
    if (i < kPadWeights) P.bf[i] = f2bf(pi);
}

// Workgroups of the backward pass: a 16-row tile a wave up to 512 waves.
static int backward_blocks(int n) { return std::min(((n + 15) / 16 + kMlpWaves - 1) / kMlpWaves, 128); }
size_t mlp_partial_floats(int n) { return (size_t)backward_blocks(n) * kMlpWaves * kPartial; }

void launch_mlp_backward(hipStream_t s, const MlpWeights& W, const float* X, const float* T, const int* idx, int n,
                         float inv_total, float* partial, const AdamArgs& P, float* loss) {
    if (n <= 0) return;
    const int blocks = backward_blocks(n);
    hipLaunchKernelGGL(k_mlp_backward, dim3(blocks), dim3(kMlpWaves * 64), 0, s, W, X, T, idx, n, inv_total, partial);
    hipLaunchKernelGGL(k_grad_apply, dim3(kPadTotal / 64 + 1), dim3(1024), 0, s, P, partial, blocks * kMlpWaves, loss);
}

__global__ void k_to_bf16(const float* p, unsigned short* bf, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) bf[i] = f2bf(p[i]);
}
void launch_to_bf16(hipStream_t s, const float* p, unsigned short* bf, int n) {
    if (n > 0) hipLaunchKernelGGL(k_to_bf16, dim3((n + 255) / 256), dim3(256), 0, s, p, bf, n);
}

// ---------------------------------------------------------------------------
// Predicted start: for a contact the plain warm start found no previous
// contact for (new this step, lambda_plain = 0), the network predicts the
// change y of slog(lambda / S), clamped to +-kMaxLogStep, so lambda =
// S sexp(slog(lambda_plain / S) + y), projected onto the friction box
// (lambda_n >= 0, |lambda_t| <= mu lambda_n).  A contact that persists keeps
// its previous-frame lambda: on a resting pile that start is already close
// to converged, closer than the network's per-contact accuracy.
AMD_INLINE double predicted(double lam_plain, double S, float y) {
    const double z = slog(lam_plain / S) + fmin(fmax((double)y, -kMaxLogStep), kMaxLogStep);
    return S * sexp(z);
}
__global__ void k_apply_prediction(ContactsView C, const BodiesView B, const float* Y, const double* scale, int n,
                                   int fric_ovr, double fric_val, double* lam_out) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    if (!C.is_new[k]) {
#pragma unroll
        for (int r = 0; r < 3; r++) lam_out[k * 3 + r] = C.lam[k * 3 + r];
        return;
    }
    double S = scale[k];
    double ln = fmax(0.0, predicted(C.lam[k * 3 + 0], S, Y[k * 3 + 0]));
    double mu;
    if (fric_ovr) {
        mu = fric_val;
    } else {
        double f1 = B.desc[C.b1[k]].friction, f2 = B.desc[C.b2[k]].friction;
        if (f1 < 0.2 || f2 < 0.2) mu = fmin(f1, f2);
        else if (f1 > 1. || f2 > 1.) mu = fmax(f1, f2);
        else mu = (f1 + f2) / 2.;
    }
    double lim = mu * ln;
    double l1 = fmin(fmax(predicted(C.lam[k * 3 + 1], S, Y[k * 3 + 1]), -lim), lim);
    double l2 = fmin(fmax(predicted(C.lam[k * 3 + 2], S, Y[k * 3 + 2]), -lim), lim);
    lam_out[k * 3 + 0] = ln;
    lam_out[k * 3 + 1] = l1;
    lam_out[k * 3 + 2] = l2;
}

void launch_apply_prediction(hipStream_t s, ContactsView C, BodiesView B, const float* Y, const double* scale, int n,
                             int fric_ovr, double fric_val, double* lam_out) {
    if (n > 0)
        hipLaunchKernelGGL(k_apply_prediction, dim3((n + 255) / 256), dim3(256), 0, s, C, B, Y, scale, n, fric_ovr,
                           fric_val, lam_out);
}

// Targets: the change of slog(lambda / S) from the plain start to the
// converged solve (features 21..23 hold the plain start's), clamped as the
// prediction is.
__global__ void k_targets(const double* lam, const double* scale, const float* X, int n, float* T) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    for (int r = 0; r < 3; r++) {
        const double d = slog(lam[k * 3 + r] / scale[k]) - (double)X[(size_t)k * kMlpIn + 21 + r];
        T[k * 3 + r] = (float)fmin(fmax(d, -kMaxLogStep), kMaxLogStep);
    }
}
void launch_targets(hipStream_t s, const double* lam, const double* scale, const float* X, int n, float* T) {
    if (n > 0) hipLaunchKernelGGL(k_targets, dim3((n + 255) / 256), dim3(256), 0, s, lam, scale, X, n, T);
}

// Start quality: with deltaV = M^-1 J^T lambda already applied (warm-start
// pass of the sweep kernel), the largest change one projected Gauss-Seidel
// row update would make, evaluated for all rows at once.
__global__ void k_start_residual(const double* rec, const int* meta, const double* dv, const double* minv,
                                 const double* jinv, int n, double omega, double compliance,
                                 unsigned long long* out) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    double r_max = 0;
    if (k < n) {
        const double* R = &rec[(size_t)k * kRecDoubles];
        int4 m = reinterpret_cast<const int4*>(meta)[k];
        const double* da = &dv[m.x * 6];
        const double* db = &dv[m.y * 6];
        double lam[3] = {R[kRecLambda], R[kRecLambda + 1], R[kRecLambda + 2]};
        for (int r = 0; r < 3; r++) {
            const double* q = R + r * kRecRow;
            const double *bv = q + kRecBv, *aw = q + kRecAw, *bw = q + kRecBw;
            double jd = (-bv[0] * da[0] + -bv[1] * da[1] + -bv[2] * da[2]) + (aw[0] * da[3] + aw[1] * da[4] + aw[2] * da[5]) +
                        (bv[0] * db[0] + bv[1] * db[1] + bv[2] * db[2]) + (bw[0] * db[3] + bw[1] * db[4] + bw[2] * db[5]);
            double D = q[kRecD];
            double l = (D * lam[r] - omega * (q[kRecB] + jd)) / (D + compliance);
            if (m.z) {
                if (r == 0) l = fmax(0.0, l);
                else l = fmin(fmax(l, -R[kRecMu] * lam[0]), R[kRecMu] * lam[0]);
            }
            r_max = fmax(r_max, fabs(l - lam[r]));
        }
    }
    for (int o = 32; o > 0; o >>= 1) r_max = fmax(r_max, __shfl_xor(r_max, o, 64));
    if ((threadIdx.x & 63) == 0 && r_max > 0) atomicMax(out, (unsigned long long)__double_as_longlong(r_max));
    (void)minv;
    (void)jinv;
}

void launch_start_residual(hipStream_t s, const double* rec, const int* meta, const double* dv, const double* minv,
                           const double* jinv, int n, double omega, double compliance, unsigned long long* out) {
    if (n > 0)
        hipLaunchKernelGGL(k_start_residual, dim3((n + 255) / 256), dim3(256), 0, s, rec, meta, dv, minv, jinv, n,
                           omega, compliance, out);
}

// lambda of the records (sweep order) <-> a list-order lambda array
__global__ void k_rec_lambda(double* rec, const int* order, const double* lam, int n, int to_rec) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int c = order[k];
    double* R = &rec[(size_t)k * kRecDoubles + kRecLambda];
    for (int r = 0; r < 3; r++) {
        if (to_rec) R[r] = lam[c * 3 + r];
    }
}
void launch_rec_lambda(hipStream_t s, double* rec, const int* order, const double* lam, int n) {
    if (n > 0) hipLaunchKernelGGL(k_rec_lambda, dim3((n + 255) / 256), dim3(256), 0, s, rec, order, lam, n, 1);
}

}  // namespace am
