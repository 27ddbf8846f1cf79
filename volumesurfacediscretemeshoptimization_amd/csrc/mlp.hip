// mlp.hip -- the learned vertex proposal: the 96-128-128-3 GELU MLP (forward,
// backward, Adam) on BF16 MFMA tiles, its training set and the one-ring
// feature encoding.
//
// There is no learned component in the reference.  The network predicts the
// displacement DMO gives a vertex (dmo/DMOTetImplCub.h:20-137,
// DMOHexImplCub.h:20-137) from its one-ring; the optimiser then searches a
// small window around the prediction and falls back to the full search.
//
// A training step is two launches: k_mlp_rows takes 16 rows per block through
// the forward and the backward pass in LDS and leaves the activations and
// their gradients feature-major, and k_mlp_grads forms the weight gradients
// (one wave per 16x16 tile, its chain over the rows in order), the bias
// gradients and the Adam update from them.  Tiles are
// __builtin_amdgcn_mfma_f32_16x16x32_bf16 (lane l: A row l%16 and B column
// l%16, k = 8*(l/16) + 0..7; D column l%16, rows 4*(l/16) + 0..3).
#include <float.h>
#include <math.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "dmo_kernels.h"
#include "mlp_internal.h"

namespace vsdmo {

__device__ __forceinline__ float gelu_d(float z)
{
    return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// Forward and backward of 16 rows per block of 4 waves.  Wave w owns the
// columns [32w, 32w + 32) of every 128-wide layer, forward and backward, so the
// pre-activations it needs for gelu' stay in its registers; A operands come
// from LDS, weight operands as 16-byte rows from global memory (W2 of the
// backward product from its transposed copy).  Outputs are feature-major
// ([feature][ld], ld = rows padded to 32): a lane's 4 rows of a column are 8
// contiguous bytes, and the weight-gradient tiles read 16 bytes along the rows.
// Rows past n are zero in X and dY.  Bound by the latency of its five layers'
// chain; 13.3 us at 4,096 rows (256 blocks, one per CU).
struct RowsArgs {
    const float* Xf;         // n x 96 rows, rounded to BF16 here, or
    const uint16_t* Xb;      // BF16 rows and targets perm[0..n) of a dataset
    const float* T;
    const int* perm;
    int n, ld;
    const uint16_t* wb;
    const uint16_t* w2t;     // W2 transposed
    const float* w;
    uint16_t *XT, *H1T, *H2T, *dZ1T, *dZ2T, *dYT;
    float* dYf;              // 3 x ld
    double* rowLoss;         // squared error of each row
};

struct RowsLds {
    MlpLds f;
    __align__(16) uint16_t dZ2[kMlpRows * kLdh];
    uint16_t dY[kMlpRows][4];
};

// 4 BF16 values of consecutive rows
__device__ __forceinline__ void store4(uint16_t* p, const uint16_t (&v)[4])
{
    *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)v[0] | (uint32_t)v[1] << 16, (uint32_t)v[2] | (uint32_t)v[3] << 16);
}

__global__ __launch_bounds__(256) void k_mlp_rows(RowsArgs a)
{
    __shared__ RowsLds sm;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r16 = lane & 15, kq = (lane >> 4) * 8, rq = (lane >> 4) * 4;
    const int row0 = blockIdx.x * kMlpRows;
    const MlpW m = mlp_load_w16(a.wb, a.w);
    if (tid < kMlpRows * (kIn / 8)) {   // 8 features per thread
        const int r = tid / (kIn / 8), c = (tid - r * (kIn / 8)) * 8;
        union { uint16_t h[8]; uint4 q; } x;
        x.q = make_uint4(0, 0, 0, 0);
        if (row0 + r < a.n) {
            if (a.Xb) {
                x.q = *reinterpret_cast<const uint4*>(a.Xb + (size_t)a.perm[row0 + r] * kIn + c);
            } else {
                const float* src = a.Xf + (size_t)(row0 + r) * kIn + c;
#pragma unroll
                for (int j = 0; j < 8; ++j) x.h[j] = f2bf(src[j]);
            }
        }
        *reinterpret_cast<uint4*>(sm.f.X + r * kLdx + c) = x.q;
    }
    // layers 2 and 3 and the backward products' operands
    bf16x8 b2[kHid / 32][2], bt[kHid / 32][2], b3[kHid / 32], b3t[2];
    const bf16x8 zero8 = __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int col = (2 * wave + t) * 16 + r16;
#pragma unroll
        for (int i = 0; i < kHid / 32; ++i) {
            b2[i][t] = *reinterpret_cast<const bf16x8*>(a.wb + kOW2 + (size_t)col * kHid + 32 * i + kq);
            bt[i][t] = *reinterpret_cast<const bf16x8*>(a.w2t + (size_t)col * kHid + 32 * i + kq);
        }
        b3t[t] = zero8;   // W3[k][col], k < 3: the first 16 lanes' first three
        if (lane < 16)
#pragma unroll
            for (int k = 0; k < kOut; ++k) b3t[t][k] = __builtin_bit_cast(__bf16, a.wb[kOW3 + k * kHid + col]);
    }
    float bias3 = 0.0f;
#pragma unroll
    for (int i = 0; i < kHid / 32; ++i) b3[i] = zero8;
    if (wave == 0 && r16 < kOut) {
#pragma unroll
        for (int i = 0; i < kHid / 32; ++i)
            b3[i] = *reinterpret_cast<const bf16x8*>(a.wb + kOW3 + (size_t)r16 * kHid + 32 * i + kq);
        bias3 = a.w[kOB3 + r16];
    }
    __syncthreads();
    for (int q = tid; q < kIn * 4; q += 256) {
        const int c = q >> 2, r = (q & 3) * 4;
        const uint16_t v[4] = { sm.f.X[r * kLdx + c], sm.f.X[(r + 1) * kLdx + c], sm.f.X[(r + 2) * kLdx + c],
                                sm.f.X[(r + 3) * kLdx + c] };
        store4(a.XT + (size_t)c * a.ld + row0 + r, v);
    }
    float z1[2][4], z2[2][4];
    // layer 1
    {
        f32x4 acc[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int i = 0; i < kIn / 32; ++i) {
            const bf16x8 av = *reinterpret_cast<const bf16x8*>(sm.f.X + r16 * kLdx + 32 * i + kq);
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, m.b1[i][t], acc[t], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int col = (2 * wave + t) * 16 + r16;
            uint16_t h[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                z1[t][r] = acc[t][r] + m.bias1[t];
                h[r] = f2bf(gelu(z1[t][r]));
                sm.f.H1[(rq + r) * kLdh + col] = h[r];
            }
            store4(a.H1T + (size_t)col * a.ld + row0 + rq, h);
        }
    }
    __syncthreads();
    // layer 2
    {
        f32x4 acc[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int i = 0; i < kHid / 32; ++i) {
            const bf16x8 av = *reinterpret_cast<const bf16x8*>(sm.f.H1 + r16 * kLdh + 32 * i + kq);
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, b2[i][t], acc[t], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int col = (2 * wave + t) * 16 + r16;
            uint16_t h[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                z2[t][r] = acc[t][r] + m.bias2[t];
                h[r] = f2bf(gelu(z2[t][r]));
                sm.f.H2[(rq + r) * kLdh + col] = h[r];
            }
            store4(a.H2T + (size_t)col * a.ld + row0 + rq, h);
        }
    }
    __syncthreads();
    // layer 3, the squared error and its gradient dY = 2 (Y - T) / n
    if (wave == 0) {
        f32x4 acc = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int i = 0; i < kHid / 32; ++i) {
            const bf16x8 av = *reinterpret_cast<const bf16x8*>(sm.f.H2 + r16 * kLdh + 32 * i + kq);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, b3[i], acc, 0, 0, 0);
        }
        if (r16 < kOut) {
#pragma unroll
            for (int r = 0; r < 4; ++r) sm.f.Y[rq + r][r16] = acc[r] + bias3;
        }
    }
    __syncthreads();
    if (tid < kMlpRows) {
        const int row = row0 + tid;
        const bool live = row < a.n;
        const size_t src = live ? (size_t)(a.Xb ? a.perm[row] : row) : 0;
        double l = 0.0;
#pragma unroll
        for (int c = 0; c < kOut; ++c) {
            float gy = 0.0f;
            if (live) {
                const float d = sm.f.Y[tid][c] - a.T[3 * src + c];
                l += (double)d * (double)d;
                gy = 2.0f * d / (float)a.n;
            }
            a.dYf[(size_t)c * a.ld + row] = gy;
            const uint16_t h = f2bf(gy);
            a.dYT[(size_t)c * a.ld + row] = h;
            sm.dY[tid][c] = h;
        }
        a.rowLoss[row] = l;
    }
    __syncthreads();
    // dZ2 = (dY W3) gelu'(Z2)
    {
        bf16x8 av = zero8;
        if (lane < 16)
#pragma unroll
            for (int k = 0; k < kOut; ++k) av[k] = __builtin_bit_cast(__bf16, sm.dY[r16][k]);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int col = (2 * wave + t) * 16 + r16;
            const f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, b3t[t], f32x4{ 0.0f, 0.0f, 0.0f, 0.0f }, 0, 0, 0);
            uint16_t h[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                h[r] = f2bf(acc[r] * gelu_d(z2[t][r]));
                sm.dZ2[(rq + r) * kLdh + col] = h[r];
            }
            store4(a.dZ2T + (size_t)col * a.ld + row0 + rq, h);
        }
    }
    __syncthreads();
    // dZ1 = (dZ2 W2) gelu'(Z1)
    {
        f32x4 acc[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int i = 0; i < kHid / 32; ++i) {
            const bf16x8 av = *reinterpret_cast<const bf16x8*>(sm.dZ2 + r16 * kLdh + 32 * i + kq);
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bt[i][t], acc[t], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int col = (2 * wave + t) * 16 + r16;
            uint16_t h[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) h[r] = f2bf(acc[t][r] * gelu_d(z1[t][r]));
            store4(a.dZ1T + (size_t)col * a.ld + row0 + rq, h);
        }
    }
}

struct GradsArgs {
    const uint16_t *XT, *H1T, *H2T, *dZ1T, *dZ2T, *dYT;
    const float* dYf;
    const double* rowLoss;
    int n, ld;
    double* part;            // squared error of every 256 rows
    float* g;                // packed gradients, or (null) the Adam update of
    float *w, *m1, *m2;
    uint16_t *wb, *w2t;
    float lr, c1, c2;
};

// the gradient gi of parameter i: stored, or Adam (beta 0.9 / 0.999, eps 1e-8)
__device__ __forceinline__ void take_grad(const GradsArgs& a, int i, float gi)
{
    if (a.g) { a.g[i] = gi; return; }
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    float m = b1 * a.m1[i] + (1.0f - b1) * gi;
    float v = b2 * a.m2[i] + (1.0f - b2) * gi * gi;
    a.m1[i] = m;
    a.m2[i] = v;
    float mh = m / a.c1, vh = v / a.c2;
    float wi = a.w[i] - a.lr * mh / (sqrtf(vh) + eps);
    a.w[i] = wi;
    const uint16_t h = f2bf(wi);
    a.wb[i] = h;
    if (i >= kOW2 && i < kOB2) a.w2t[((i - kOW2) & (kHid - 1)) * kHid + ((i - kOW2) >> 7)] = h;
}

// the weight-gradient tiles of dW2, dW1 and dW3
constexpr int kTiles2 = (kHid / 16) * (kHid / 16), kTiles1 = (kHid / 16) * (kIn / 16), kTiles3 = kHid / 16;
constexpr int kTiles = kTiles2 + kTiles1 + kTiles3, kCols = 2 * kHid + kOut;

// dW = dZ^T H and the bias gradients of one step, one wave per block: the
// first kTiles blocks one 16x16 tile each, accumulated over the rows in order
// (32 per MFMA, the next kAhead x 32 rows' operands in flight; the same sums as
// a product per layer), the next kCols blocks a column sum each (256 strided
// FP64 sums, then a fixed tree), the others the squared error of 256 rows each.
// Bound by the loads' latency: 12.7 us at 4,096 rows (8, 12, 16 and 24 steps in
// flight measure the same; the column sums with 2-byte loads 23 us).  The two
// launches replace 16 per step (a product per layer and direction with strided
// 2-byte operand loads), 370 us at 4,096 rows.
__global__ __launch_bounds__(64) void k_mlp_grads(GradsArgs a)
{
    const int lane = threadIdx.x;
    int b = blockIdx.x;
    if (b < kTiles) {
        const int r16 = lane & 15, kq = (lane >> 4) * 8;
        const uint16_t *A, *B;
        int off, ldg, mt, nt, rows = kHid;
        if (b < kTiles2) {
            A = a.dZ2T; B = a.H1T; off = kOW2; ldg = kHid;
            mt = b / (kHid / 16); nt = b % (kHid / 16);
        } else if (b < kTiles2 + kTiles1) {
            b -= kTiles2;
            A = a.dZ1T; B = a.XT; off = kOW1; ldg = kIn;
            mt = b / (kIn / 16); nt = b % (kIn / 16);
        } else {
            A = a.dYT; B = a.H2T; off = kOW3; ldg = kHid; rows = kOut;
            mt = 0; nt = b - kTiles2 - kTiles1;
        }
        const bool has = mt * 16 + r16 < rows;
        const uint16_t* pa = A + (size_t)(has ? mt * 16 + r16 : 0) * a.ld + kq;
        const uint16_t* pb = B + (size_t)(nt * 16 + r16) * a.ld + kq;
        f32x4 acc = { 0.0f, 0.0f, 0.0f, 0.0f };
        constexpr int kAhead = 8;
        const int steps = a.ld / 32;
        const bf16x8 zero8 = __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
        bf16x8 va[2][kAhead], vb[2][kAhead];
        auto load = [&](int s0, bf16x8 (&x)[kAhead], bf16x8 (&y)[kAhead]) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int s = s0 + u < steps ? s0 + u : steps - 1;
                x[u] = *reinterpret_cast<const bf16x8*>(pa + 32 * s);
                y[u] = *reinterpret_cast<const bf16x8*>(pb + 32 * s);
            }
        };
        auto mul = [&](int s0, const bf16x8 (&x)[kAhead], const bf16x8 (&y)[kAhead]) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
                if (s0 + u < steps) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(has ? x[u] : zero8, y[u], acc, 0, 0, 0);
        };
        load(0, va[0], vb[0]);
        for (int s = 0; s < steps; s += 2 * kAhead) {
            load(s + kAhead, va[1], vb[1]);
            mul(s, va[0], vb[0]);
            load(s + 2 * kAhead, va[0], vb[0]);
            mul(s + kAhead, va[1], vb[1]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int mrow = mt * 16 + 4 * (lane >> 4) + r;
            if (mrow < rows) take_grad(a, off + mrow * ldg + nt * 16 + r16, acc[r]);
        }
        return;
    }
    __shared__ double s[256];
    b -= kTiles;
    auto tree = [&]() {
        __syncthreads();
        for (int k = 128; k > 0; k >>= 1) {
            for (int t = lane; t < k; t += 64) s[t] += s[t + k];
            __syncthreads();
        }
    };
    if (b < kCols) {
        // sum t takes rows t, t + 256, ...; lane l < 32 holds sums 8l..8l+7, so
        // that its loads are 16 bytes (rows past n are zero)
        if (lane < 32) {
            double acc[8] = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
            if (b < 2 * kHid) {
                const uint16_t* col = (b < kHid ? a.dZ1T + (size_t)b * a.ld : a.dZ2T + (size_t)(b - kHid) * a.ld);
#pragma unroll 8
                for (int r = 8 * lane; r < a.ld; r += 256) {
                    union { uint4 q; uint16_t h[8]; } v;
                    v.q = *reinterpret_cast<const uint4*>(col + r);
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[j] += (double)bf2f(v.h[j]);
                }
            } else {
                const float* col = a.dYf + (size_t)(b - 2 * kHid) * a.ld;
#pragma unroll 4
                for (int r = 8 * lane; r < a.ld; r += 256) {
                    const float4 u = *reinterpret_cast<const float4*>(col + r), v = *reinterpret_cast<const float4*>(col + r + 4);
                    acc[0] += (double)u.x; acc[1] += (double)u.y; acc[2] += (double)u.z; acc[3] += (double)u.w;
                    acc[4] += (double)v.x; acc[5] += (double)v.y; acc[6] += (double)v.z; acc[7] += (double)v.w;
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) s[8 * lane + j] = acc[j];
        }
        tree();
        if (lane == 0)
            take_grad(a, b < kHid ? kOB1 + b : b < 2 * kHid ? kOB2 + b - kHid : kOB3 + b - 2 * kHid, (float)s[0]);
        return;
    }
    b -= kCols;
    for (int t = lane; t < 256; t += 64) {
        const int r = b * 256 + t;
        s[t] = r < a.n ? a.rowLoss[r] : 0.0;
    }
    tree();
    if (lane == 0) a.part[b] = s[0];
}

// mean loss of `steps` batches of n rows, from the nb partial sums of each
// (one thread, fixed order)
__global__ void k_loss_final(const double* __restrict__ part, int nb, int n, int steps, double* __restrict__ out)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double acc = 0.0;
    for (int st = 0; st < steps; ++st) {
        double s = 0.0;
        for (int i = 0; i < nb; ++i) s += part[(size_t)st * nb + i];
        acc += s / (double)n;
    }
    *out = acc;
}

__global__ void k_to_bf16(const float* __restrict__ a, long long n, uint16_t* __restrict__ b)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = f2bf(a[i]);
}

// BF16 copy of W2, transposed
__global__ void k_w2_transposed(const uint16_t* __restrict__ wb, uint16_t* __restrict__ w2t)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kHid * kHid) w2t[(i & (kHid - 1)) * kHid + (i >> 7)] = wb[kOW2 + i];
}

// one-ring features of vertex v into o[0..95] (bf16); returns L
__device__ __forceinline__ float vertex_features(const float* __restrict__ x, const float* __restrict__ y,
                                                 const float* __restrict__ z, const int* __restrict__ nbr, int v,
                                                 uint16_t* o)
{
    const int* nb = nbr + (size_t)v * kNbr;
    const float vx = x[v], vy = y[v], vz = z[v];
    float sum = 0.0f;
    int cnt = 0;
    for (int k = 0; k < kNbr; ++k) {
        int u = nb[k];
        if (u < 0) break;
        float dx = x[u] - vx, dy = y[u] - vy, dz = z[u] - vz;
        sum += sqrtf((dx * dx + dy * dy) + dz * dz);
        ++cnt;
    }
    float l = cnt > 0 ? sum / (float)cnt : 1.0f;
    if (!(l > 0.0f)) l = 1.0f;
    for (int k = 0; k < kNbr; ++k) {
        int u = nb[k];
        if (u < 0) {
            o[3 * k] = 0; o[3 * k + 1] = 0; o[3 * k + 2] = 0;
        } else {
            o[3 * k] = f2bf((x[u] - vx) / l);
            o[3 * k + 1] = f2bf((y[u] - vy) / l);
            o[3 * k + 2] = f2bf((z[u] - vz) / l);
        }
    }
    return l;
}

// one-ring features: thread per vertex
__global__ void k_features(const float* __restrict__ x, const float* __restrict__ y, const float* __restrict__ z,
                           const int* __restrict__ nbr, int lo, int hi, uint16_t* __restrict__ X, float* __restrict__ L,
                           float* __restrict__ v0)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int v = lo + i;
    if (v >= hi) return;
    L[i] = vertex_features(x, y, z, nbr, v, X + (size_t)i * kIn);
    v0[3 * i] = x[v]; v0[3 * i + 1] = y[v]; v0[3 * i + 2] = z[v];
}

struct InferArgs {
    const float* x;
    const float* y;
    const float* z;
    const int* nbr;
    int lo, n;
    const float* Xin;      // optional precomputed features (n x 96, rounded to BF16 here)
    const uint16_t* wb;
    const float* w;
    float* Y;
    float* L;
};

// Fused inference, 16 rows per block of 4 waves (mlp_features16 /
// mlp_layers16): features (from the positions, or rows of Xin) -> LDS, the
// three layers on MFMA tiles.  Writes Y and L of rows [0, n).
__global__ __launch_bounds__(256) void k_mlp_infer(InferArgs a)
{
    __shared__ MlpLds sm;
    const int tid = threadIdx.x;
    const int row0 = blockIdx.x * kMlpRows;
    if (a.Xin) {
        for (int i = tid; i < kMlpRows * kIn; i += 256) {
            int r = i / kIn, c = i - r * kIn;
            sm.X[r * kLdx + c] = (row0 + r < a.n) ? f2bf(a.Xin[(size_t)(row0 + r) * kIn + c]) : (uint16_t)0;
        }
    } else {
        const int r = tid >> 4;
        const bool live = row0 + r < a.n;
        mlp_features16(a.x, a.y, a.z, a.nbr, a.lo + row0 + r, live, sm);
        if (live && (tid & 15) == 0) a.L[row0 + r] = sm.L[r];
    }
    __syncthreads();
    mlp_layers16(a.wb, a.w, sm);
    if (tid < kMlpRows * kOut) {
        const int r = tid / kOut, o = tid - r * kOut;
        if (row0 + r < a.n) a.Y[(size_t)(row0 + r) * kOut + o] = sm.Y[r][o];
    }
}

void launch_mlp_infer(vsdmo_mlp* m, const float* x, const float* y, const float* z, const int* nbr, int lo, int hi,
                      const float* Xin, float* Y, float* L, hipStream_t s)
{
    const int n = hi - lo;
    if (n <= 0) return;
    InferArgs a{ x, y, z, nbr, lo, n, Xin, m->wb.p, m->w.p, Y, L };
    k_mlp_infer<<<(n + kMlpRows - 1) / kMlpRows, 256, 0, s>>>(a);
}

__global__ void k_targets(const float* __restrict__ x, const float* __restrict__ y, const float* __restrict__ z, int lo,
                          int hi, const float* __restrict__ L, const float* __restrict__ v0, float* __restrict__ T)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int v = lo + i;
    if (v >= hi) return;
    const float l = L[i];
    T[3 * i] = (x[v] - v0[3 * i]) / l;
    T[3 * i + 1] = (y[v] - v0[3 * i + 1]) / l;
    T[3 * i + 2] = (z[v] - v0[3 * i + 2]) / l;
}

void launch_features(const float* x, const float* y, const float* z, const int* nbr, int lo, int hi, uint16_t* X,
                     float* L, float* v0, hipStream_t s)
{
    if (hi > lo) k_features<<<(hi - lo + 127) / 128, 128, 0, s>>>(x, y, z, nbr, lo, hi, X, L, v0);
}

void launch_targets(const float* x, const float* y, const float* z, int lo, int hi, const float* L, const float* v0,
                    float* T, hipStream_t s)
{
    if (hi > lo) k_targets<<<(hi - lo + 127) / 128, 128, 0, s>>>(x, y, z, lo, hi, L, v0, T);
}

// Neighbour table of the vertices from lo on (the distinct corners of the ring
// in order of first appearance, up to kNbr, then -1) and the place in it of
// every ring corner (kRingLocNone: a corner beyond the table, padding, the
// rings of vertices before lo).  A wave per vertex, lane q holding entry q: the
// ring's corners are loaded 64 at a time, and every turn places the first corner
// left and all its repeats, so a ring takes as many turns as it has distinct
// corners (14 in a tet cube, 26 in a hex cube).  Bound by latency, not by the
// 30-50 MB that it moves: 32 us for the 40^3 tet cube, 60 us for the 48^3 hex cube.
// The proposal's first setting on a mesh takes 0.48 / 0.52 ms by it (allocations),
// with the table built on the host 12.3 / 18.7 ms.
__global__ __launch_bounds__(256) void k_neighbour_table(const int* __restrict__ row, const int* __restrict__ val, int nV,
                                                         int lo, int st, int ls, int* __restrict__ nbr,
                                                         uint8_t* __restrict__ loc)
{
    const int v = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
    const int lane = threadIdx.x & 63;
    if (v >= nV) return;
    const int e0 = row[v];
    const int n = (row[v + 1] - e0) * ls;
    int o = -1, cnt = 0;
    for (int base = 0; base < n; base += 64) {
        const int j = base + lane, e = j / ls, k = j - e * ls;
        const bool in = v >= lo && j < n && k < st;
        const int u = in ? val[(size_t)(e0 + e) * st + k] : -1;
        int q = kRingLocNone;
        unsigned long long left = __ballot(in);
        while (left) {
            const int w = __builtin_amdgcn_readlane(u, __builtin_ctzll(left));
            const unsigned long long known = __ballot(o == w);
            int at = kRingLocNone;
            if (known) at = __builtin_ctzll(known);
            else if (cnt < kNbr) {
                at = cnt++;
                if (lane == at) o = w;
            }
            if (u == w) q = at;
            left &= ~__ballot(u == w);
        }
        if (j < n) loc[(size_t)e0 * ls + j] = (uint8_t)q;
    }
    if (lane < kNbr) nbr[(size_t)v * kNbr + lane] = o;
}

void build_neighbour_table(vsdmo_mesh& m)
{
    if (m.nbr.p) return;
    const int st = (m.elem == VSDMO_TET) ? 3 : 7;
    const int ls = (m.elem == VSDMO_TET) ? kRingLocStrideTet : kRingLocStrideHex;
    m.ringLoc.alloc(std::max<size_t>(m.ringVal.n / st * ls, 1));
    m.nbr.alloc((size_t)m.nV * kNbr);
    if (m.nV > 0)
        k_neighbour_table<<<(m.nV + 3) / 4, 256, 0, m.stream>>>(m.ringRow.p, m.ringVal.p, m.nV, m.nSurf, st, ls, m.nbr.p,
                                                                m.ringLoc.p);
    VSDMO_HIP(hipGetLastError());
    VSDMO_HIP(hipStreamSynchronize(m.stream));
}

void mlp_reserve(vsdmo_mlp* m, int n)
{
    if (n <= m->cap) return;
    const size_t c = (size_t)(std::max(n, 2 * m->cap) + 31) / 32 * 32;
    m->XT.alloc(c * kIn);
    m->H1T.alloc(c * kHid);
    m->H2T.alloc(c * kHid);
    m->dZ1T.alloc(c * kHid);
    m->dZ2T.alloc(c * kHid);
    m->dYT.alloc(c * kOut);
    m->dYf.alloc(c * kOut);
    m->rowLoss.alloc(c);
    m->cap = (int)c;
}

// n rows of features and targets: FP32 rows, or rows perm[0..n) of a dataset
struct MlpBatch {
    const float* Xf = nullptr;
    const uint16_t* Xb = nullptr;
    const float* T = nullptr;
    const int* perm = nullptr;
    int n = 0;
};

// forward, backward and the weight gradients of a batch; the squared error of
// every 256 rows in part; gradients in m->g, or (adam) the update of step
// m->step with rate lr
static void mlp_step(vsdmo_mlp* m, const MlpBatch& x, double* part, bool adam, float lr, hipStream_t s)
{
    const int ld = (x.n + 31) / 32 * 32;
    k_mlp_rows<<<ld / kMlpRows, 256, 0, s>>>(RowsArgs{ x.Xf, x.Xb, x.T, x.perm, x.n, ld, m->wb.p, m->w2t.p, m->w.p, m->XT.p,
                                                      m->H1T.p, m->H2T.p, m->dZ1T.p, m->dZ2T.p, m->dYT.p, m->dYf.p,
                                                      m->rowLoss.p });
    GradsArgs g{ m->XT.p, m->H1T.p, m->H2T.p, m->dZ1T.p, m->dZ2T.p, m->dYT.p, m->dYf.p, m->rowLoss.p, x.n, ld, part,
                 adam ? nullptr : m->g.p, m->w.p, m->m1.p, m->m2.p, m->wb.p, m->w2t.p, lr, 1.0f, 1.0f };
    if (adam) {
        g.c1 = 1.0f - std::pow(0.9f, (float)m->step);
        g.c2 = 1.0f - std::pow(0.999f, (float)m->step);
    }
    k_mlp_grads<<<kTiles + kCols + (x.n + 255) / 256, 64, 0, s>>>(g);
}

static void refresh_bf16(vsdmo_mlp* m, hipStream_t s)
{
    k_to_bf16<<<(kNParams + 255) / 256, 256, 0, s>>>(m->w.p, kNParams, m->wb.p);
    k_w2_transposed<<<kHid * kHid / 256, 256, 0, s>>>(m->wb.p, m->w2t.p);
}

static vsdmo_status fail_m(vsdmo_status st, const std::string& msg)
{
    set_error(msg);
    return st;
}

template <class F>
static vsdmo_status guarded_m(F&& f)
{
    try {
        return f();
    } catch (const HipError& e) {
        return fail_m(VSDMO_HIP_ERROR, std::string(hipGetErrorString(e.code)) + " in " + e.where);
    } catch (const StatusError& e) {
        return fail_m(e.status, e.msg);
    } catch (const std::bad_alloc&) {
        return fail_m(VSDMO_HIP_ERROR, "host allocation failed");
    }
}

// the FP32 rows and targets of the host calls
static void reserve_rows(vsdmo_mlp* m, int n)
{
    if (m->Xf.n < (size_t)n * kIn) m->Xf.alloc((size_t)n * kIn);
    if (m->T.n < (size_t)n * kOut) m->T.alloc((size_t)n * kOut);
}

static uint64_t smix(uint64_t& s)
{
    uint64_t z = (s += 0x9e3779b97f4a7c15ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

}  // namespace vsdmo

using namespace vsdmo;

extern "C" {

int32_t vsdmo_mlp_num_params(void) { return kNParams; }

vsdmo_status vsdmo_mlp_create(uint64_t seed, vsdmo_mlp** out)
{
    return guarded_m([&]() -> vsdmo_status {
        if (!out) return fail_m(VSDMO_INVALID_ARG, "out is NULL");
        *out = nullptr;
        auto* m = new vsdmo_mlp();
        try {
            VSDMO_HIP(hipStreamCreate(&m->stream));
            // uniform(-1/sqrt(fan_in), 1/sqrt(fan_in)) for weights and biases
            std::vector<float> w(kNParams);
            uint64_t s = seed;
            auto fill = [&](int off, int cnt, int fan) {
                float b = 1.0f / std::sqrt((float)fan);
                for (int i = 0; i < cnt; ++i) {
                    double u = (double)(smix(s) >> 11) * (1.0 / 9007199254740992.0);
                    w[off + i] = (float)((2.0 * u - 1.0) * b);
                }
            };
            fill(kOW1, kHid * kIn, kIn); fill(kOB1, kHid, kIn);
            fill(kOW2, kHid * kHid, kHid); fill(kOB2, kHid, kHid);
            fill(kOW3, kOut * kHid, kHid); fill(kOB3, kOut, kHid);
            m->w.alloc(kNParams); m->g.alloc(kNParams); m->m1.alloc(kNParams); m->m2.alloc(kNParams);
            m->wb.alloc(kNParams);
            m->w2t.alloc((size_t)kHid * kHid);
            m->w.upload(w.data(), kNParams, m->stream);
            std::vector<float> zero(kNParams, 0.0f);
            m->m1.upload(zero.data(), kNParams, m->stream);
            m->m2.upload(zero.data(), kNParams, m->stream);
            refresh_bf16(m, m->stream);
            VSDMO_HIP(hipStreamSynchronize(m->stream));
        } catch (...) {
            if (m->stream) (void)hipStreamDestroy(m->stream);
            delete m;
            throw;
        }
        *out = m;
        return VSDMO_OK;
    });
}

vsdmo_status vsdmo_mlp_destroy(vsdmo_mlp* m)
{
    if (!m) return VSDMO_OK;
    if (m->n_users > 0)
        return fail_m(VSDMO_INVALID_ARG, "network still set as the proposal of an optimiser or batch");
    if (m->stream) {
        (void)hipStreamSynchronize(m->stream);
        (void)hipStreamDestroy(m->stream);
    }
    delete m;
    return VSDMO_OK;
}

vsdmo_status vsdmo_mlp_get_params(vsdmo_mlp* m, float* out)
{
    return guarded_m([&]() -> vsdmo_status {
        if (!m || !out) return fail_m(VSDMO_INVALID_ARG, "NULL argument");
        m->w.download(out, kNParams, m->stream);
        VSDMO_HIP(hipStreamSynchronize(m->stream));
        return VSDMO_OK;
    });
}

vsdmo_status vsdmo_mlp_set_params(vsdmo_mlp* m, const float* in)
{
    return guarded_m([&]() -> vsdmo_status {
        if (!m || !in) return fail_m(VSDMO_INVALID_ARG, "NULL argument");
        m->w.upload(in, kNParams, m->stream);
        refresh_bf16(m, m->stream);
        std::vector<float> zero(kNParams, 0.0f);
        m->m1.upload(zero.data(), kNParams, m->stream);
        m->m2.upload(zero.data(), kNParams, m->stream);
        m->step = 0;
        VSDMO_HIP(hipStreamSynchronize(m->stream));
        return VSDMO_OK;
    });
}

vsdmo_status vsdmo_mlp_forward(vsdmo_mlp* m, const float* X, int32_t n, float* Y)
{
    return guarded_m([&]() -> vsdmo_status {
        if (!m || !X || !Y || n < 0) return fail_m(VSDMO_INVALID_ARG, "bad argument");
        if (n == 0) return VSDMO_OK;
        reserve_rows(m, n);
        m->Xf.upload(X, (size_t)n * kIn, m->stream);
        launch_mlp_infer(m, nullptr, nullptr, nullptr, nullptr, 0, n, m->Xf.p, m->T.p, nullptr, m->stream);
        m->T.download(Y, (size_t)n * kOut, m->stream);
        VSDMO_HIP(hipStreamSynchronize(m->stream));
        return VSDMO_OK;
    });
}

vsdmo_status vsdmo_mlp_gradients(vsdmo_mlp* m, const float* X, const float* T, int32_t n, double* loss, float* grad)
{
    return guarded_m([&]() -> vsdmo_status {
        if (!m || !X || !T || n <= 0) return fail_m(VSDMO_INVALID_ARG, "bad argument");
        mlp_reserve(m, n);
        reserve_rows(m, n);
        m->Xf.upload(X, (size_t)n * kIn, m->stream);
        m->T.upload(T, (size_t)n * kOut, m->stream);
        const int nb = (n + 255) / 256;
        DevBuf<double> part((size_t)nb + 1);   // partial sums, then the loss
        MlpBatch x;
        x.Xf = m->Xf.p; x.T = m->T.p; x.n = n;
        mlp_step(m, x, part.p, false, 0.0f, m->stream);
        k_loss_final<<<1, 64, 0, m->stream>>>(part.p, nb, n, 1, part.p + nb);
        VSDMO_HIP(hipGetLastError());
        if (grad) m->g.download(grad, kNParams, m->stream);
        double l = 0.0;
        VSDMO_HIP(hipMemcpyAsync(&l, part.p + nb, sizeof(double), hipMemcpyDeviceToHost, m->stream));
        VSDMO_HIP(hipStreamSynchronize(m->stream));
        if (loss) *loss = l;
        return VSDMO_OK;
    });
}

vsdmo_status vsdmo_mlp_train(vsdmo_mlp* m, vsdmo_dataset* ds, int32_t epochs, int32_t batch, float lr, uint64_t seed,
                             double* epoch_loss)
{
    return guarded_m([&]() -> vsdmo_status {
        if (!m || !ds) return fail_m(VSDMO_INVALID_ARG, "NULL argument");
        if (epochs < 0 || batch <= 0 || !(lr > 0.0f)) return fail_m(VSDMO_INVALID_ARG, "bad training parameters");
        const long long N = ds->n;
        if (N < batch) return fail_m(VSDMO_INVALID_ARG, "dataset smaller than one batch");
        if (N >= (1LL << 31)) return fail_m(VSDMO_INVALID_ARG, "dataset too large");
        hipStream_t s = m->stream;
        VSDMO_HIP(hipStreamSynchronize(ds->stream));
        mlp_reserve(m, batch);
        if (epochs == 0) return VSDMO_OK;
        m->perm.alloc((size_t)N);
        const long long steps = N / batch;   // the ragged tail of each shuffled epoch is dropped
        const int nb = (batch + 255) / 256;
        DevBuf<double> part((size_t)steps * nb), loss((size_t)epochs);
        // the host shuffles an epoch while the GPU runs the one before: two
        // permutations in turn, each free again once its upload is done
        std::vector<int> perm[2] = { std::vector<int>((size_t)N), std::vector<int>((size_t)N) };
        struct Events {
            hipEvent_t e[2] = { nullptr, nullptr };
            ~Events() { for (hipEvent_t x : e) if (x) (void)hipEventDestroy(x); }
        } up;
        struct Drain {   // an early exit must not free what the stream still reads
            hipStream_t s;
            ~Drain() { (void)hipStreamSynchronize(s); }
        } drain{ s };
        for (hipEvent_t& e : up.e) VSDMO_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        uint64_t rs = seed;
        for (int ep = 0; ep < epochs; ++ep) {
            std::vector<int>& p = perm[ep & 1];
            if (ep >= 2) VSDMO_HIP(hipEventSynchronize(up.e[ep & 1]));
            for (long long i = 0; i < N; ++i) p[i] = (int)i;
            for (long long i = N - 1; i > 0; --i) std::swap(p[i], p[(long long)(smix(rs) % (uint64_t)(i + 1))]);
            m->perm.upload(p.data(), (size_t)N, s);
            VSDMO_HIP(hipEventRecord(up.e[ep & 1], s));
            for (long long st = 0; st < steps; ++st) {
                MlpBatch x;
                x.Xb = ds->X.p; x.T = ds->T.p; x.perm = m->perm.p + st * batch; x.n = batch;
                m->step++;
                mlp_step(m, x, part.p + st * nb, true, lr, s);
            }
            k_loss_final<<<1, 64, 0, s>>>(part.p, nb, batch, (int)steps, loss.p + ep);
        }
        std::vector<double> l((size_t)epochs);
        loss.download(l.data(), (size_t)epochs, s);
        VSDMO_HIP(hipStreamSynchronize(s));
        if (epoch_loss)
            for (int ep = 0; ep < epochs; ++ep) epoch_loss[ep] = l[ep] / (double)steps;
        VSDMO_HIP(hipGetLastError());
        return VSDMO_OK;
    });
}

vsdmo_status vsdmo_dataset_create(int64_t capacity, vsdmo_dataset** out)
{
    return guarded_m([&]() -> vsdmo_status {
        if (!out || capacity <= 0) return fail_m(VSDMO_INVALID_ARG, "bad argument");
        *out = nullptr;
        auto* d = new vsdmo_dataset();
        try {
            VSDMO_HIP(hipStreamCreate(&d->stream));
            d->cap = capacity;
            d->X.alloc((size_t)capacity * kIn);
            d->T.alloc((size_t)capacity * kOut);
        } catch (...) {
            if (d->stream) (void)hipStreamDestroy(d->stream);
            delete d;
            throw;
        }
        *out = d;
        return VSDMO_OK;
    });
}

vsdmo_status vsdmo_dataset_size(vsdmo_dataset* d, int64_t* n)
{
    if (!d || !n) return fail_m(VSDMO_INVALID_ARG, "NULL argument");
    *n = d->n;
    return VSDMO_OK;
}

vsdmo_status vsdmo_dataset_get(vsdmo_dataset* d, int64_t start, int32_t n, float* X, float* T)
{
    return guarded_m([&]() -> vsdmo_status {
        if (!d || start < 0 || n < 0 || start + n > d->n) return fail_m(VSDMO_INVALID_ARG, "range outside the dataset");
        if (X) {
            std::vector<uint16_t> xb((size_t)n * kIn);
            VSDMO_HIP(hipMemcpyAsync(xb.data(), d->X.p + start * kIn, xb.size() * 2, hipMemcpyDeviceToHost, d->stream));
            VSDMO_HIP(hipStreamSynchronize(d->stream));
            for (size_t i = 0; i < xb.size(); ++i) X[i] = bf2f(xb[i]);
        }
        if (T) {
            VSDMO_HIP(hipMemcpyAsync(T, d->T.p + start * kOut, sizeof(float) * n * kOut, hipMemcpyDeviceToHost, d->stream));
            VSDMO_HIP(hipStreamSynchronize(d->stream));
        }
        return VSDMO_OK;
    });
}

vsdmo_status vsdmo_dataset_destroy(vsdmo_dataset* d)
{
    if (!d) return VSDMO_OK;
    if (d->stream) {
        (void)hipStreamSynchronize(d->stream);
        (void)hipStreamDestroy(d->stream);
    }
    delete d;
    return VSDMO_OK;
}

}  // extern "C"
