// Learned saddle proposal on gfx950: symmetry-function descriptors and the
// MLP 48 -> 128 -> 128 -> 3 (SiLU) with hand-written BF16 MFMA forward and
// backward GEMMs, FP32 accumulation, FP32 master weights and Adam.
//
// GEMM tiles: one wavefront computes 16 x 16 output tiles with
// v_mfma_f32_16x16x16_bf16 (lane l holds A[l%16][4(l/16)..+3],
// B[4(l/16)..+3][l%16] and D[4(l/16)..+3][l%16]).  Activations are FP32 in
// registers and rounded to BF16 (round to nearest even) as MFMA operands.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "akmc_internal.h"

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kB = 256;

__device__ inline uint16_t to_bf16(float f)
{
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ inline float sigm(float z) { return 1.0f / (1.0f + __expf(-z)); }

// The network 48 -> 128 -> 128 -> 3 and its flat parameter layout
constexpr int kIn = 48, kHid = 128, kOut = 3;
constexpr int kW1 = 0, kB1 = kIn * kHid, kW2 = kB1 + kHid, kB2 = kW2 + kHid * kHid, kW3 = kB2 + kHid,
              kB3 = kW3 + kHid * kOut, kParam = kB3 + kOut;
static_assert(kParam == AKMC_MLP_PARAMS, "parameter count");

constexpr int kTile = 64;      // rows of a forward workgroup, 16 per wavefront
constexpr int kRP = kHid + 4;  // pitch of row-major BF16 operands in LDS

__device__ inline f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }
__device__ inline bf16x4 bf4(const uint16_t *p) { return *reinterpret_cast<const bf16x4 *>(p); }
// the operand of 16 rows of X (48 inputs) per lane: X[row][16 s + lk ..+3]
__device__ inline void load_rows(const float *X, long long row, bool ok, int lk, bf16x4 (&a)[3])
{
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        const float4 v = ok ? *reinterpret_cast<const float4 *>(X + row * kIn + 16 * s + lk) : make_float4(0, 0, 0, 0);
        a[s] = bf16x4{(short)to_bf16(v.x), (short)to_bf16(v.y), (short)to_bf16(v.z), (short)to_bf16(v.w)};
    }
}

// Weights are stored in the order the matrix instruction reads them: the
// operand B[k][n] of column tile nt and k-step s is 64 lanes x 4 values, so a
// wavefront's load is 512 contiguous bytes (as rows of W^T it touched 16
// lines: the loads, not the products, set the pace)
__host__ __device__ constexpr int frag(int n, int k, int ks)
{
    return (((n / 16) * ks + k / 16) * 64 + (k % 16) / 4 * 16 + n % 16) * 4 + k % 4;
}
__device__ inline bf16x4 wfrag(const uint16_t *w, int nt, int s, int ks)
{
    return bf4(w + ((nt * ks + s) * 64 + (threadIdx.x & 63)) * 4);
}

// one hidden layer of the wavefront's 16 rows: Z = A W + b into registers,
// silu(Z) as BF16 row-major (hr) and per column tile to put(tile, 4 rows)
template <int KS, typename PUT>
__device__ inline void hidden_layer(const bf16x4 (&a)[KS], const uint16_t *wt, const float *bias, int r0, int li, int lk,
                                    f32x4 (&Z)[8], uint16_t (*hr)[kRP], PUT put)
{
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
        const int col = 16 * nt + li;
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < KS; ++s) acc = mfma(a[s], wfrag(wt, nt, s, KS), acc);
        const float bb = bias[col];
        bf16x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float z = acc[e] + bb;
            Z[nt][e] = z;
            h[e] = (short)to_bf16(z * sigm(z));
            hr[r0 + lk + e][col] = (uint16_t)h[e];
        }
        put(nt, h);
        // a few column tiles' weights in flight, not all eight: registers
        if (nt % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
}

// Y [M][3] = network(X [M][48])
__global__ void __launch_bounds__(kB) k_mlp_forward(const float *__restrict__ X, int M, const float *__restrict__ p,
                                                    const uint16_t *__restrict__ w1t, const uint16_t *__restrict__ w2t,
                                                    const uint16_t *__restrict__ w3t, float *__restrict__ Y)
{
    __shared__ uint16_t h1[kTile][kRP], h2[kTile][kRP];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r0 = 16 * wave;
    const int li = lane & 15, lk = (lane >> 4) * 4;
    const long long m0 = (long long)blockIdx.x * kTile;
    bf16x4 a1[3], a[8];
    f32x4 Z[8];
    load_rows(X, m0 + r0 + li, m0 + r0 + li < M, lk, a1);
    hidden_layer<3>(a1, w1t, p + kB1, r0, li, lk, Z, h1, [](int, bf16x4) {});
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 8; ++s) a[s] = bf4(&h1[r0 + li][16 * s + lk]);
    hidden_layer<8>(a, w2t, p + kB2, r0, li, lk, Z, h2, [](int, bf16x4) {});
    __syncthreads();
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 8; ++s) acc = mfma(bf4(&h2[r0 + li][16 * s + lk]), wfrag(w3t, 0, s, 8), acc);
    if (li >= kOut) return;
    const float bb = p[kB3 + li];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const long long row = m0 + r0 + lk + e;
        if (row < M) Y[row * kOut + li] = acc[e] + bb;
    }
}

// Gradient of the mean-squared loss over rows idx[0 .. M) of (X, T) (idx
// null: rows 0 .. M), in an order of summation that depends on M alone:
// weight gradients over kChunk rows at a time by one matrix-instruction chain
// each, the chunks in order; bias gradients as the sums over the rows equal
// modulo kChunk, in order, and a tree over these.
//
// k_mlp_rows: one wavefront per 16 rows, forward and backward.  What the
// weight gradients contract over the rows goes to memory in the order the
// matrix instruction reads it (MlpRows: a 16-row x 16-column tile is 64 lanes
// x 4 rows, 512 contiguous bytes in BF16).  k_mlp_wgrad: per chunk 96
// wavefronts, one per 16 x 16 tile of dW1, dW2, dW3, and a workgroup per 16
// bias columns.  Bound by latency at 4096 rows: 25 us (256 wavefronts, one per
// CU, each through five dependent layers of 512-byte weight loads) and 14 us
// (a bias sum is a chain over the chunks).  Forward and backward of 4096 rows
// 35 us in all; 91 us with a launch per layer, 41 us as one kernel that also
// summed the weight gradients, in another order.
constexpr int kChunk = 256;  // rows of a weight-gradient partial sum

struct MlpRows {
    uint16_t *x, *h1, *h2;  // [row tile][column tile][64][4] BF16: inputs, activations
    float *z1, *z2;         // the same in FP32: d loss / d pre-activation
    float *r;               // [row tile][64][4]: Y - T, 3 of 16 columns
};

__global__ void __launch_bounds__(64) k_mlp_rows(const float *__restrict__ X, const float *__restrict__ T,
                                                 const int *__restrict__ idx, int M, const float *__restrict__ p,
                                                 const uint16_t *__restrict__ w1t, const uint16_t *__restrict__ w2t,
                                                 const uint16_t *__restrict__ w3t, const uint16_t *__restrict__ w2r,
                                                 const uint16_t *__restrict__ w3r, MlpRows o)
{
    __shared__ uint16_t hr[16][kRP], h2r[16][kRP];  // H1, then dZ2; H2
    __shared__ uint16_t xt[kIn][20], yr[16][20];    // X transposed; dY
    const int lane = threadIdx.x, li = lane & 15, lk = (lane >> 4) * 4;
    const size_t tile = blockIdx.x;
    const int m0 = 16 * blockIdx.x;
    f32x4 Z1[8], Z2[8];
    // rows past M have no part in the sums: zeros
    auto put = [&](uint16_t *dst, int nt, bf16x4 v) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (m0 + lk + e >= M) v[e] = 0;
        *reinterpret_cast<bf16x4 *>(dst + ((tile * 8 + nt) * 64 + lane) * 4) = v;
    };
    {
        bf16x4 a[3];
        const bool ok = m0 + li < M;
        load_rows(X, ok ? (idx ? idx[m0 + li] : m0 + li) : 0, ok, lk, a);
#pragma unroll
        for (int s = 0; s < 3; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) xt[16 * s + lk + e][li] = (uint16_t)a[s][e];
        hidden_layer<3>(a, w1t, p + kB1, 0, li, lk, Z1, hr, [&](int nt, bf16x4 h) { put(o.h1, nt, h); });
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 3; ++s)
        *reinterpret_cast<bf16x4 *>(o.x + ((tile * 3 + s) * 64 + lane) * 4) = bf4(&xt[16 * s + li][lk]);
    {
        bf16x4 a[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) a[s] = bf4(&hr[li][16 * s + lk]);
        hidden_layer<8>(a, w2t, p + kB2, 0, li, lk, Z2, h2r, [&](int nt, bf16x4 h) { put(o.h2, nt, h); });
    }
    __syncthreads();
    {
        // output layer, error r = Y - T and dY = 2 r / M
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, r = acc;
#pragma unroll
        for (int s = 0; s < 8; ++s) acc = mfma(bf4(&h2r[li][16 * s + lk]), wfrag(w3t, 0, s, 8), acc);
        const float bb = li < kOut ? p[kB3 + li] : 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = m0 + lk + e;
            if (m < M && li < kOut) r[e] = acc[e] + bb - T[(long long)(idx ? idx[m] : m) * kOut + li];
            yr[lk + e][li] = to_bf16(2.0f * r[e] / (float)M);
        }
        *reinterpret_cast<f32x4 *>(o.r + (tile * 64 + lane) * 4) = r;
    }
    __syncthreads();
    {
        const bf16x4 a = bf4(&yr[li][lk]);
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            f32x4 v = mfma(a, wfrag(w3r, nt, 0, 1), f32x4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float z = Z2[nt][e], s = sigm(z);
                v[e] = m0 + lk + e < M ? v[e] * s * (1.0f + z * (1.0f - s)) : 0.0f;
                hr[lk + e][16 * nt + li] = to_bf16(v[e]);
            }
            *reinterpret_cast<f32x4 *>(o.z2 + ((tile * 8 + nt) * 64 + lane) * 4) = v;
        }
    }
    __syncthreads();
    {
        bf16x4 a[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) a[s] = bf4(&hr[li][16 * s + lk]);
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < 8; ++s) v = mfma(a[s], wfrag(w2r, nt, s, 8), v);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float z = Z1[nt][e], s = sigm(z);
                v[e] = m0 + lk + e < M ? v[e] * s * (1.0f + z * (1.0f - s)) : 0.0f;
            }
            *reinterpret_cast<f32x4 *>(o.z1 + ((tile * 8 + nt) * 64 + lane) * 4) = v;
            if (nt % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

__device__ inline bf16x4 bf16_of(f32x4 v)
{
    return bf16x4{(short)to_bf16(v[0]), (short)to_bf16(v[1]), (short)to_bf16(v[2]), (short)to_bf16(v[3])};
}

// Per chunk seven workgroups of 16 wavefronts: six with a 16 x 16 tile of the
// weight gradients per wavefront (P [chunk][kParam]) and one for the squared
// error (part [chunk]); after them one per 16 bias columns (into g)
constexpr int kWgBlock = 1024, kWgPer = 7;
constexpr int kWgBias = 17;  // dZ1, dZ2 (8 column tiles each), dY
__global__ void __launch_bounds__(kWgBlock) k_mlp_wgrad(MlpRows in, int M, int nchunk, float *__restrict__ P,
                                                        double *__restrict__ part, float *__restrict__ g)
{
    constexpr int kTiles = kChunk / 16;  // row tiles of a chunk
    __shared__ double sh[kChunk * 17 / 2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lk = (lane >> 4) * 4;
    const int ntile = (M + 15) / 16;
    auto frag4 = [&](const float *src, size_t t) { return *reinterpret_cast<const f32x4 *>(src + (t * 64 + lane) * 4); };
    auto dy = [&](f32x4 r) {
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = 2.0f * r[e] / (float)M;
        return r;
    };
    if ((int)blockIdx.x < kWgPer * nchunk) {
        const int chunk = blockIdx.x / kWgPer, part_of = blockIdx.x % kWgPer;
        const int t0 = chunk * kTiles, t1 = min(t0 + kTiles, ntile);
        if (part_of == kWgPer - 1) {
            if (tid < kChunk) {
                double l = 0.0;
                const int m = chunk * kChunk + tid;
                if (m < M)
                    for (int c = 0; c < kOut; ++c) {
                        const float r = in.r[((size_t)(m / 16) * 64 + (m % 16) / 4 * 16 + c) * 4 + m % 4];
                        l += (double)r * r;
                    }
                sh[tid] = l;
            }
            __syncthreads();
            for (int o = kChunk / 2; o > 0; o >>= 1) {
                if (tid < o) sh[tid] += sh[tid + o];
                __syncthreads();
            }
            if (tid == 0) part[chunk] = sh[0];
            return;
        }
        // tiles 0 .. 63: dW2, 64 .. 87: dW1, 88 .. 95: dW3
        const int t = part_of * (kWgBlock / 64) + wave;
        const int kind = t < 64 ? 0 : t < 88 ? 1 : 2, u = kind == 0 ? t : kind == 1 ? t - 64 : t - 88;
        const int i = kind == 2 ? u : u / 8, j = kind == 2 ? 0 : u % 8, an = kind == 1 ? 3 : 8;
        const uint16_t *A = kind == 0 ? in.h1 : kind == 1 ? in.x : in.h2;
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int r0 = t0; r0 < t1; r0 += 4) {  // four row tiles' operands in flight
            bf16x4 a[4];
            f32x4 v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const size_t rt = min(r0 + q, t1 - 1);
                a[q] = bf4(A + ((rt * an + i) * 64 + lane) * 4);
                v[q] = kind == 0 ? frag4(in.z2, rt * 8 + j) : kind == 1 ? frag4(in.z1, rt * 8 + j) : dy(frag4(in.r, rt));
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (r0 + q < t1) acc = mfma(a[q], bf16_of(v[q]), acc);
        }
        float *out = P + (size_t)chunk * kParam;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = 16 * i + lk + e;
            if (kind == 0) out[kW2 + k * kHid + 16 * j + li] = acc[e];
            else if (kind == 1) out[kW1 + k * kHid + 16 * j + li] = acc[e];
            else if (li < kOut) out[kW3 + k * kOut + li] = acc[e];
        }
        return;
    }
    // column sums: wavefront v holds the rows 16 v .. 16 v + 15 modulo kChunk
    const int bt = blockIdx.x - kWgPer * nchunk, j = bt % 8;
    float (*tree)[17] = reinterpret_cast<float (*)[17]>(sh);
    f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int rt = wave; rt < ntile; rt += kTiles)
        s += bt < 8 ? frag4(in.z1, (size_t)rt * 8 + j) : bt < 16 ? frag4(in.z2, (size_t)rt * 8 + j) : dy(frag4(in.r, rt));
#pragma unroll
    for (int e = 0; e < 4; ++e) tree[16 * wave + lk + e][li] = s[e];
    __syncthreads();
    for (int o = kChunk / 2; o > 0; o >>= 1) {
        for (int q = tid; q < o * 16; q += kWgBlock) tree[q / 16][q % 16] += tree[q / 16 + o][q % 16];
        __syncthreads();
    }
    if (tid < (bt < 16 ? 16 : kOut)) g[(bt < 8 ? kB1 + 16 * j : bt < 16 ? kB2 + 16 * j : kB3) + tid] = tree[0][tid];
}

// BF16 copies of parameter i in fragment order: the forward operands
// B[k][n] = W[k][n] and the backward-data ones B[n][k] = W[k][n], the output
// layer padded to 16
struct MlpBf16 {
    uint16_t *w1t, *w2t, *w3t, *w2r, *w3r;
};
__device__ inline void store_bf16(const MlpBf16 &w, int i, float v)
{
    const uint16_t h = to_bf16(v);
    if (i < kB1) {
        w.w1t[frag(i % kHid, i / kHid, 3)] = h;
    } else if (i >= kW2 && i < kB2) {
        const int t = i - kW2;
        w.w2t[frag(t % kHid, t / kHid, 8)] = h;
        w.w2r[frag(t / kHid, t % kHid, 8)] = h;
    } else if (i >= kW3 && i < kB3) {
        const int t = i - kW3;
        w.w3t[frag(t % kOut, t / kOut, 8)] = h;
        w.w3r[frag(t / kOut, t % kOut, 1)] = h;
    }
}

__global__ void k_weights_bf16(const float *__restrict__ p, MlpBf16 w)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 16 * kHid) {  // the padding of the output layer
        const int k = i / 16, n = i % 16;
        if (n >= kOut) {
            w.w3t[frag(n, k, 8)] = 0;
            w.w3r[frag(k, n, 1)] = 0;
        }
    }
    if (i < kParam) store_bf16(w, i, p[i]);
}

// the weights' gradient: the chunks' sums in order (the biases' is in g
// already); with step the Adam step and the BF16 copies of the parameter; the
// loss of the rows, scaled, is added to acc
constexpr int kUpd = 128;  // parameters per workgroup
__global__ void __launch_bounds__(kUpd) k_mlp_update(const float *__restrict__ P, int nchunk, float *__restrict__ g,
                                                     float *__restrict__ p, float *__restrict__ m1,
                                                     float *__restrict__ m2, MlpBf16 w, int step, float lr, float b1,
                                                     float b2, float eps, float c1, float c2,
                                                     const double *__restrict__ part, double scale,
                                                     double *__restrict__ acc)
{
    const int i = blockIdx.x * kUpd + threadIdx.x;
    if (i < kParam) {
        const bool bias = (i >= kB1 && i < kW2) || (i >= kB2 && i < kW3) || i >= kB3;
        float gi = 0.0f;
        if (bias) {
            gi = g[i];
        } else {
#pragma unroll 8
            for (int c = 0; c < nchunk; ++c) gi += P[(size_t)c * kParam + i];
            g[i] = gi;
        }
        if (step) {
            const float a = b1 * m1[i] + (1.0f - b1) * gi;
            const float b = b2 * m2[i] + (1.0f - b2) * gi * gi;
            m1[i] = a;
            m2[i] = b;
            const float v = p[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
            p[i] = v;
            store_bf16(w, i, v);
        }
    }
    if (acc && blockIdx.x == 0 && threadIdx.x == kUpd - 1) {
        double t = 0.0;
        for (int c = 0; c < nchunk; ++c) t += part[c];
        *acc += t * scale;
    }
}

// X = (X - mean) * scale, feature by feature, in FP32
__global__ void k_standardize(float *__restrict__ X, long long n, const float *__restrict__ mean,
                              const float *__restrict__ scale)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int c = int(t % kIn);
    X[t] = __fmul_rn(__fsub_rn(X[t], mean[c]), scale[c]);
}

// ------------------------------------------------------------ descriptors

__device__ inline float fcut(float r, float rc) { return r < rc ? 0.5f * (__cosf(3.14159265f * r / rc) + 1.0f) : 0.0f; }

// The 48 descriptors of a query (atom, vacancy site, candidate mover): 32
// radial G2 (16 over the atoms, 8 over the vacancy site and 8 over the mover
// as pseudo-neighbours of their own kinds) and 16 angular G4; the definitions
// are restated in FP64 by the test oracle.  The 32 terms over the atoms do
// not depend on the site and mover, and a proposal asks for the same free
// atoms with every mover, so k_atom_descriptors computes them once per atom
// and k_query_descriptors assembles the queries.
constexpr float kDescRc = 7.22f, kDescRca = 5.0f;
constexpr int kDescCap = AKMC_DESC_CAP;  // neighbours inside kDescRca kept in LDS at most

// sum over the wavefront, the same bits on every lane
__device__ inline float wave_sum(float v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// One wavefront per atom, neighbours from the walker's list at its resident
// positions (minimum image).  Radial terms: neighbours 64 at a time, one per
// lane, their (r, fc) passed round in LDS so that lane l sums centre l % 16
// over every fourth neighbour.  Angular terms: the neighbours inside 5 A are
// compacted into LDS in list order and their pairs dealt to the lanes.
// Bound by exp and the vector instructions of the pair terms: 9,600 atoms
// with 134 neighbours and 42 inside 5 A each take 123 us, and the
// 252,000 queries' rows 66 us, where a thread per query took 16.7 ms.
__global__ void __launch_bounds__(64) k_atom_descriptors(BatchDev b, int na, const int *__restrict__ atoms, int cap,
                                                         float *__restrict__ G)
{
    extern __shared__ float4 ang[];  // [cap] x, y, z, r of the angular neighbours
    __shared__ float sr[64], sf[64];
    const int q = blockIdx.x, lane = threadIdx.x;
    const int i = atoms[q];
    const WalkerDev W = b.walkers[b.wk[i]];
    const double4 pi = b.p4[i];
    const int cnt = b.nnb[i];
    float *fa = reinterpret_cast<float *>(ang + cap);  // [cap] fc(r, 5 A)
    const float centre = 2.0f + 5.0f * (lane & 15) / 15.0f;
    float g2 = 0.0f;
    int m = 0;
    for (int k0 = 0; k0 < cnt; k0 += 64) {
        float r = 0.0f, ax = 0.0f, ay = 0.0f, az = 0.0f;
        bool in = false;
        if (k0 + lane < cnt) {
            const uint32_t e = nbr_entry(b, k0 + lane, i);
            const double4 pj = b.p4[W.off + int(e & AKMC_NB_JMASK)];
            double dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
            dx -= W.L[0] * rint(dx * W.invL[0]);
            dy -= W.L[1] * rint(dy * W.invL[1]);
            dz -= W.L[2] * rint(dz * W.invL[2]);
            r = (float)sqrt(dx * dx + dy * dy + dz * dz);
            in = !(r < 1.0e-8f || r >= kDescRc);
            ax = (float)dx;
            ay = (float)dy;
            az = (float)dz;
        }
        const unsigned long long bal = __ballot(in);
        const int at = __popcll(bal & ((1ull << lane) - 1ull)), n = __popcll(bal);
        __syncthreads();  // the previous round's (r, fc) are read
        if (in) {
            sr[at] = r;
            sf[at] = fcut(r, kDescRc);
        }
        const bool near = in && r < kDescRca;
        const unsigned long long baln = __ballot(near);
        const int an = m + __popcll(baln & ((1ull << lane) - 1ull));
        if (near && an < cap) {
            ang[an] = make_float4(ax, ay, az, r);
            fa[an] = fcut(r, kDescRca);
        }
        m += __popcll(baln);
        __syncthreads();
        for (int t = lane >> 4; t < n; t += 4) {
            const float d = sr[t] - centre;
            g2 += __expf(-8.0f * d * d) * sf[t];
        }
    }
    g2 += __shfl_xor(g2, 16);
    g2 += __shfl_xor(g2, 32);
    if (m > cap) {
        if (lane == 0) atomicOr(b.overflow, AKMC_OV_LIST);
        m = cap;
    }
    float g[16];
    for (int t = 0; t < 16; ++t) g[t] = 0.0f;
    // pair p of the m (m - 1) / 2 pairs j < k, row after row (row j starts at
    // j (2m - j - 1) / 2), dealt to the lanes in turn
    const int total = m * (m - 1) / 2;
    for (int p = lane; p < total; p += 64) {
        const float h = 2.0f * m - 1.0f;
        int j = int(0.5f * (h - sqrtf(fmaxf(h * h - 8.0f * p, 0.0f))));
        j = min(max(j, 0), m - 2);
        while (j > 0 && j * (2 * m - j - 1) / 2 > p) --j;  // the float root may be a row off
        while ((j + 1) * (2 * m - j - 2) / 2 <= p) ++j;
        const int k = j + 1 + p - j * (2 * m - j - 1) / 2;
        const float4 a = ang[j];
        const float faj = fa[j];
        const float4 c = ang[k];
        const float bx = c.x - a.x, by = c.y - a.y, bz = c.z - a.z;
        const float rjk = sqrtf(bx * bx + by * by + bz * bz);
        if (rjk >= kDescRca) continue;
        const float base = faj * fa[k] * fcut(rjk, kDescRca);
        const float cs = (a.x * c.x + a.y * c.y + a.z * c.z) / (a.w * c.w);
        const float rr = a.w * a.w + c.w * c.w + rjk * rjk;
        const float x0 = __expf(-0.005f * rr) * base, x1 = __expf(-0.02f * rr) * base;
#pragma unroll
        for (int li = 0; li < 2; ++li) {
            const float c1 = 1.0f + (li == 0 ? cs : -cs);
            const float c2 = c1 * c1, c4 = c2 * c2, c8 = c4 * c4;
            // zeta 1, 2, 4, 16; 2^(1 - zeta) is exact and applied at the end
            const float pw[4] = {c1, c2, c4, c8 * c8};
#pragma unroll
            for (int z = 0; z < 4; ++z) {
                g[4 * z + 2 * li] += pw[z] * x0;
                g[4 * z + 2 * li + 1] += pw[z] * x1;
            }
        }
    }
    float out = lane < 16 ? g2 : 0.0f;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        const float v = wave_sum(g[t]) * (t < 4 ? 1.0f : t < 8 ? 0.5f : t < 12 ? 0.125f : 3.0517578125e-5f);
        if (lane == 16 + t) out = v;
    }
    if (lane < 32) G[(size_t)q * 32 + lane] = out;
}

// a query's row: its atom's 32 terms and the radial terms of the vacancy
// site and the mover, one thread per element
__global__ void __launch_bounds__(kB) k_query_descriptors(BatchDev b, int nq, const int *__restrict__ qatom,
                                                          const int *__restrict__ qslot,
                                                          const double *__restrict__ qvac,
                                                          const double *__restrict__ qmov, const float *__restrict__ G,
                                                          float *__restrict__ X)
{
    const long long t = (long long)blockIdx.x * kB + threadIdx.x;
    if (t >= 48ll * nq) return;
    const int q = int(t / 48), c = int(t - 48ll * q);
    float v;
    if (c < 16 || c >= 32) {
        v = G[(size_t)qslot[q] * 32 + (c < 16 ? c : c - 16)];
    } else {
        const int i = qatom[q];
        const WalkerDev &W = b.walkers[b.wk[i]];
        const double4 pi = b.p4[i];
        const double *u = (c < 24 ? qvac : qmov) + 3ll * q;
        const double pp[3] = {pi.x, pi.y, pi.z};
        double d2 = 0.0;
        for (int a = 0; a < 3; ++a) {
            double d = pp[a] - u[a];
            d -= W.L[a] * rint(d * W.invL[a]);
            d2 += d * d;
        }
        const float r = (float)sqrt(d2);
        const int k = c & 7;
        const float s = r - (c < 24 ? 1.5f + 5.0f * k / 7.0f : 6.0f * k / 7.0f);
        v = __expf(-2.0f * s * s) * fcut(r, kDescRc);
    }
    X[t] = v;
}

}  // namespace

// ------------------------------------------------------------ launchers

void akmc_mlp_launch_weights(const float *p, uint16_t *w1t, uint16_t *w2t, uint16_t *w3t, uint16_t *w2r,
                             uint16_t *w3r, hipStream_t s)
{
    k_weights_bf16<<<(kParam + kB - 1) / kB, kB, 0, s>>>(p, MlpBf16{w1t, w2t, w3t, w2r, w3r});
}

void akmc_mlp_launch_standardize(float *X, long long rows, const float *mean, const float *scale, hipStream_t s)
{
    k_standardize<<<(unsigned)((rows * kIn + kB - 1) / kB), kB, 0, s>>>(X, rows * kIn, mean, scale);
}

void akmc_mlp_launch_forward(const float *X, int M, const float *p, const uint16_t *w1t, const uint16_t *w2t,
                             const uint16_t *w3t, float *Y, hipStream_t s)
{
    k_mlp_forward<<<(M + kTile - 1) / kTile, kB, 0, s>>>(X, M, p, w1t, w2t, w3t, Y);
}

int akmc_mlp_grad_chunks(int M) { return (M + kChunk - 1) / kChunk; }

size_t akmc_mlp_rows_bytes(int rows)
{
    const size_t tiles = (rows + 15) / 16;
    return tiles * 64 * 4 * ((3 + 8 + 8) * sizeof(uint16_t) + (8 + 8 + 1) * sizeof(float));
}

void akmc_mlp_launch_grad(const float *X, const float *T, const int *idx, int M, const float *p, const uint16_t *w1t,
                          const uint16_t *w2t, const uint16_t *w3t, const uint16_t *w2r, const uint16_t *w3r,
                          void *rows, float *P, double *part, float *g, hipStream_t s)
{
    const int tiles = (M + 15) / 16, nchunk = akmc_mlp_grad_chunks(M);
    const size_t t = (size_t)tiles * 64 * 4;
    MlpRows o;
    o.z1 = (float *)rows;
    o.z2 = o.z1 + 8 * t;
    o.r = o.z2 + 8 * t;
    o.h1 = (uint16_t *)(o.r + t);
    o.h2 = o.h1 + 8 * t;
    o.x = o.h2 + 8 * t;
    k_mlp_rows<<<tiles, 64, 0, s>>>(X, T, idx, M, p, w1t, w2t, w3t, w2r, w3r, o);
    k_mlp_wgrad<<<kWgPer * nchunk + kWgBias, kWgBlock, 0, s>>>(o, M, nchunk, P, part, g);
}

void akmc_mlp_launch_update(const float *P, int M, float *g, float *p, float *m1, float *m2, uint16_t *w1t,
                            uint16_t *w2t, uint16_t *w3t, uint16_t *w2r, uint16_t *w3r, int step, float lr, int t,
                            const double *part, double *acc, hipStream_t s)
{
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
    k_mlp_update<<<(kParam + kUpd - 1) / kUpd, kUpd, 0, s>>>(P, akmc_mlp_grad_chunks(M), g, p, m1, m2,
                                                             MlpBf16{w1t, w2t, w3t, w2r, w3r}, step, lr, b1, b2,
                                                             1.0e-8f, c1, c2, part, 1.0 / M, acc);
}

void akmc_mlp_launch_descriptors(const BatchDev &b, int na, const int *atoms, int nq, const int *qatom,
                                 const int *qslot, const double *qvac, const double *qmov, float *G, float *X,
                                 hipStream_t s)
{
    const int cap = b.maxnb < kDescCap ? b.maxnb : kDescCap;
    k_atom_descriptors<<<na, 64, (size_t)cap * 20, s>>>(b, na, atoms, cap, G);
    k_query_descriptors<<<(unsigned)((48ll * nq + kB - 1) / kB), kB, 0, s>>>(b, nq, qatom, qslot, qvac, qmov, G, X);
}
