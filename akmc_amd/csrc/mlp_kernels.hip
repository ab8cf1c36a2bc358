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

// Forward and backward of a tile of 64 rows stay in one workgroup: wavefront
// v takes rows 16 v .. 16 v + 15 through every layer (its pre-activations
// stay in registers for the backward pass), activations pass from layer to
// layer through LDS as the BF16 operands of the next product, row-major for
// the layers and transposed for the weight gradients.  Before, each layer
// was a launch that wrote its FP32 activations to memory: 17 launches per
// minibatch, most of them launch latency at 4096 rows.
constexpr int kTile = 64;
constexpr int kTP = kTile + 4;  // pitch of the transposed operands (BF16), rows of 8-byte multiples
constexpr int kRP = kHid + 4;   // pitch of the row-major ones

struct MlpLds {
    uint16_t xt[kIn][kTP], h1t[kHid][kTP], h2t[kHid][kTP], z1t[kHid][kTP], z2t[kHid][kTP], yt[16][kTP];
    uint16_t hr[kTile][kRP];   // H1, then dZ2, row-major
    uint16_t h2r[kTile][kRP];
    uint16_t yr[kTile][20];    // dY
    float bsum[4][2 * kHid + 16];  // per wavefront: column sums of dZ1, dZ2, dY
    double loss[4];
};

__device__ inline f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }
__device__ inline bf16x4 bf4(const uint16_t *p) { return *reinterpret_cast<const bf16x4 *>(p); }
__device__ inline float dsilu(float z)
{
    const float s = sigm(z);
    return s * (1.0f + z * (1.0f - s));
}

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
// silu(Z) as BF16 row-major (hr) and, when TR, transposed (ht)
template <int KS, bool TR>
__device__ inline void hidden_layer(const bf16x4 (&a)[KS], const uint16_t *wt, const float *bias, int r0, int li, int lk,
                                    f32x4 (&Z)[8], uint16_t (*hr)[kRP], uint16_t (*ht)[kTP])
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
        if constexpr (TR) *reinterpret_cast<bf16x4 *>(&ht[col][r0 + lk]) = h;
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
    hidden_layer<3, false>(a1, w1t, p + kB1, r0, li, lk, Z, h1, nullptr);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 8; ++s) a[s] = bf4(&h1[r0 + li][16 * s + lk]);
    hidden_layer<8, false>(a, w2t, p + kB2, r0, li, lk, Z, h2, nullptr);
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
// null: rows 0 .. M): the tiles of a workgroup add up in registers, its sums
// go to P[blockIdx.x][kParam] and its squared error to part[blockIdx.x]
__global__ void __launch_bounds__(kB, 1) k_mlp_grad(const float *__restrict__ X, const float *__restrict__ T,
                                                 const int *__restrict__ idx, int M, const float *__restrict__ p,
                                                 const uint16_t *__restrict__ w1t, const uint16_t *__restrict__ w2t,
                                                 const uint16_t *__restrict__ w3t, const uint16_t *__restrict__ w2r,
                                                 const uint16_t *__restrict__ w3r, float *__restrict__ P,
                                                 double *__restrict__ part)
{
    __shared__ MlpLds L;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int r0 = 16 * wave, li = lane & 15, lk = (lane >> 4) * 4;
    f32x4 g1[6], g2[16], g3[2];  // this wavefront's tiles of dW1, dW2, dW3
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    for (auto &v : g1) v = zero;
    for (auto &v : g2) v = zero;
    for (auto &v : g3) v = zero;
    float s1[8] = {}, s2[8] = {}, s3 = 0.0f;  // column sums of dZ1, dZ2, dY
    double sq = 0.0;
    const int ntiles = (M + kTile - 1) / kTile;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int m0 = tile * kTile;
        __syncthreads();  // the previous tile's operands are read
        // (the LDS addresses below are not worth a register each across tiles)
        asm volatile("" : "+v"(r0), "+v"(li), "+v"(lk));
        f32x4 Z1[8], Z2[8];
        {
            bf16x4 a[3];
            const int m = m0 + r0 + li;
            const bool ok = m < M;
            load_rows(X, ok ? (idx ? idx[m] : m) : 0, ok, lk, a);
#pragma unroll
            for (int s = 0; s < 3; ++s)
#pragma unroll
                for (int e = 0; e < 4; ++e) L.xt[16 * s + lk + e][r0 + li] = (uint16_t)a[s][e];
            hidden_layer<3, true>(a, w1t, p + kB1, r0, li, lk, Z1, L.hr, L.h1t);
        }
        __syncthreads();
        {
            bf16x4 a[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) a[s] = bf4(&L.hr[r0 + li][16 * s + lk]);
            hidden_layer<8, true>(a, w2t, p + kB2, r0, li, lk, Z2, L.h2r, L.h2t);
        }
        __syncthreads();
        {
            // output layer, error and dY = 2 (Y - T) / M; rows past M have none
            f32x4 acc = zero;
#pragma unroll
            for (int s = 0; s < 8; ++s) acc = mfma(bf4(&L.h2r[r0 + li][16 * s + lk]), wfrag(w3t, 0, s, 8), acc);
            const float bb = li < kOut ? p[kB3 + li] : 0.0f;
            bf16x4 d;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + r0 + lk + e;
                float r = 0.0f;
                if (m < M && li < kOut) r = acc[e] + bb - T[(long long)(idx ? idx[m] : m) * kOut + li];
                sq += (double)r * r;
                const float dy = 2.0f * r / (float)M;
                s3 += dy;
                d[e] = (short)to_bf16(dy);
                L.yr[r0 + lk + e][li] = (uint16_t)d[e];
            }
            *reinterpret_cast<bf16x4 *>(&L.yt[li][r0 + lk]) = d;
        }
        __syncthreads();
        {
            const bf16x4 a = bf4(&L.yr[r0 + li][lk]);
#pragma unroll
            for (int nt = 0; nt < 8; ++nt) {
                const int col = 16 * nt + li;
                const f32x4 acc = mfma(a, wfrag(w3r, nt, 0, 1), zero);
                bf16x4 d;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v = acc[e] * dsilu(Z2[nt][e]);
                    s2[nt] += v;
                    d[e] = (short)to_bf16(v);
                    L.hr[r0 + lk + e][col] = (uint16_t)d[e];
                }
                *reinterpret_cast<bf16x4 *>(&L.z2t[col][r0 + lk]) = d;
            }
        }
        __syncthreads();
        {
            bf16x4 a[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) a[s] = bf4(&L.hr[r0 + li][16 * s + lk]);
#pragma unroll
            for (int nt = 0; nt < 8; ++nt) {
                const int col = 16 * nt + li;
                f32x4 acc = zero;
#pragma unroll
                for (int s = 0; s < 8; ++s) acc = mfma(a[s], wfrag(w2r, nt, s, 8), acc);
                bf16x4 d;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v = acc[e] * dsilu(Z1[nt][e]);
                    s1[nt] += v;
                    d[e] = (short)to_bf16(v);
                }
                *reinterpret_cast<bf16x4 *>(&L.z1t[col][r0 + lk]) = d;
                if (nt % 2 == 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
        // weight gradients over the tile's 64 rows: wavefront v takes row
        // tiles 2 v, 2 v + 1 of dW2 and dW3 and the tiles 6 v .. 6 v + 5 of dW1
#pragma unroll 1
        for (int s = 0; s < 4; ++s) {
            const int m = 16 * s + lk;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const bf16x4 a = bf4(&L.h1t[16 * (2 * wave + i) + li][m]);
#pragma unroll
                for (int j = 0; j < 8; ++j) g2[8 * i + j] = mfma(a, bf4(&L.z2t[16 * j + li][m]), g2[8 * i + j]);
                g3[i] = mfma(bf4(&L.h2t[16 * (2 * wave + i) + li][m]), bf4(&L.yt[li][m]), g3[i]);
            }
#pragma unroll
            for (int t = 0; t < 6; ++t) {
                const int i = (6 * wave + t) / 8, j = (6 * wave + t) % 8;
                g1[t] = mfma(bf4(&L.xt[16 * i + li][m]), bf4(&L.z1t[16 * j + li][m]), g1[t]);
            }
        }
    }
    float *out = P + (size_t)blockIdx.x * kParam;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int k = 16 * (2 * wave + i) + lk + e;
#pragma unroll
            for (int j = 0; j < 8; ++j) out[kW2 + k * kHid + 16 * j + li] = g2[8 * i + j][e];
            if (li < kOut) out[kW3 + k * kOut + li] = g3[i][e];
        }
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            const int i = (6 * wave + t) / 8, j = (6 * wave + t) % 8;
            out[kW1 + (16 * i + lk + e) * kHid + 16 * j + li] = g1[t][e];
        }
    }
    // column sums: the four row groups of a wavefront, then the wavefronts in order
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
        s1[nt] += __shfl_xor(s1[nt], 16);
        s1[nt] += __shfl_xor(s1[nt], 32);
        s2[nt] += __shfl_xor(s2[nt], 16);
        s2[nt] += __shfl_xor(s2[nt], 32);
    }
    s3 += __shfl_xor(s3, 16);
    s3 += __shfl_xor(s3, 32);
    for (int o = 1; o < 64; o <<= 1) sq += __shfl_xor(sq, o);
    if (lane < 16) {
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            L.bsum[wave][16 * nt + li] = s1[nt];
            L.bsum[wave][kHid + 16 * nt + li] = s2[nt];
        }
        L.bsum[wave][2 * kHid + li] = s3;
    }
    if (lane == 0) L.loss[wave] = sq;
    __syncthreads();
    for (int c = threadIdx.x; c < 2 * kHid + kOut; c += kB) {
        const float v = ((L.bsum[0][c] + L.bsum[1][c]) + L.bsum[2][c]) + L.bsum[3][c];
        out[c < kHid ? kB1 + c : c < 2 * kHid ? kB2 + c - kHid : kB3 + c - 2 * kHid] = v;
    }
    if (threadIdx.x == 0) part[blockIdx.x] = ((L.loss[0] + L.loss[1]) + L.loss[2]) + L.loss[3];
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

// the gradient: the workgroups' sums in order, four interleaved runs of them
// per parameter added in a fixed order; with step the Adam step and the
// BF16 copies of the parameter; the loss of the rows, scaled, is added to acc
constexpr int kUpd = 64;  // parameters per workgroup
__global__ void __launch_bounds__(4 * kUpd) k_mlp_update(const float *__restrict__ P, int nb, float *__restrict__ g,
                                                         float *__restrict__ p, float *__restrict__ m1,
                                                         float *__restrict__ m2, MlpBf16 w, int step, float lr, float b1, float b2,
                                                         float eps, float c1, float c2, const double *__restrict__ part,
                                                         double scale, double *__restrict__ acc)
{
    __shared__ float sh[4][kUpd];
    const int c = threadIdx.x % kUpd, run = threadIdx.x / kUpd, i = blockIdx.x * kUpd + c;
    float s = 0.0f;
    if (i < kParam)
        for (int k = run; k < nb; k += 4) s += P[(size_t)k * kParam + i];
    sh[run][c] = s;
    __syncthreads();
    if (run == 0 && i < kParam) {
        const float gi = (sh[0][c] + sh[1][c]) + (sh[2][c] + sh[3][c]);
        g[i] = gi;
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
    if (acc && blockIdx.x == 0 && threadIdx.x == 4 * kUpd - 1) {
        double t = 0.0;
        for (int k = 0; k < nb; ++k) t += part[k];
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
constexpr int kDescCap = 4096;  // neighbours inside kDescRca kept in LDS at most

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

int akmc_mlp_grad_blocks(int M)
{
    const int tiles = (M + kTile - 1) / kTile;
    return tiles < AKMC_MLP_MAXBLOCKS ? tiles : AKMC_MLP_MAXBLOCKS;
}

void akmc_mlp_launch_grad(const float *X, const float *T, const int *idx, int M, const float *p, const uint16_t *w1t,
                          const uint16_t *w2t, const uint16_t *w3t, const uint16_t *w2r, const uint16_t *w3r, float *P,
                          double *part, hipStream_t s)
{
    k_mlp_grad<<<akmc_mlp_grad_blocks(M), kB, 0, s>>>(X, T, idx, M, p, w1t, w2t, w3t, w2r, w3r, P, part);
}

void akmc_mlp_launch_update(const float *P, int M, float *g, float *p, float *m1, float *m2, uint16_t *w1t,
                            uint16_t *w2t, uint16_t *w3t, uint16_t *w2r, uint16_t *w3r, int step, float lr, int t,
                            const double *part, double *acc, hipStream_t s)
{
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
    k_mlp_update<<<(kParam + kUpd - 1) / kUpd, 4 * kUpd, 0, s>>>(P, akmc_mlp_grad_blocks(M), g, p, m1, m2,
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
