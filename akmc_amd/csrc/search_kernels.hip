// Kernels of the walker state machines (search_logic.h): the logic kernel,
// walker starts, probes and harvests.
#include "search_logic.h"

namespace {

// a walker in the loop of a plain FIRE relax with every atom free, which
// k_relax_fire advances
__device__ inline bool fire_walker(const SearchDev &s, const WalkerState &w, int n, int nact)
{
    return s.fire_on && w.kind == WK_RELAX && w.state == ST_R_STEP && nact == n && n <= AKMC_FIRE_ATOMS;
}

#if AKMC_LOGIC_BLOCK == 256
// One iteration of FIRE (relax_logic's step of optim/Relax.cpp:44-315 for
// semi-implicit Euler without frozen atoms) per launch: one workgroup per
// walker, up to kFireAtoms of its atoms per thread, whose force, velocity
// and position stay in registers between the two block sums (centre-of-mass
// velocity; powers and norms).  Bound by memory: each atom's force, velocity
// and position are read once and velocity, position and probe written once,
// 144 bytes.  512 walkers, 1.07 M atoms: 76 us where the general state machine,
// reading them in every pass, took 143 us.
constexpr int kFireBlock = 1024, kFireWaves = kFireBlock / 64;
constexpr int kFireAtoms = AKMC_FIRE_ATOMS / kFireBlock;

template <int NV>
__device__ inline void fire_sum(double (&v)[NV], double *sh)
{
#pragma unroll
    for (int c = 0; c < NV; ++c)
        for (int o = 32; o > 0; o >>= 1) v[c] += __shfl_xor(v[c], o);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int c = 0; c < NV; ++c) sh[c * kFireWaves + (threadIdx.x >> 6)] = v[c];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NV; ++c) {
        double t = sh[c * kFireWaves];
        for (int k = 1; k < kFireWaves; ++k) t += sh[c * kFireWaves + k];
        v[c] = t;
    }
    __syncthreads();
}

__global__ void __launch_bounds__(kFireBlock) k_relax_fire(BatchDev b, SearchDev s)
{
    __shared__ double sh[4 * kFireWaves];
    const int wid = blockIdx.x, tid = threadIdx.x;
    const WalkerDev &W = b.walkers[wid];
    const int off = W.off, n = W.n;
    const size_t A = b.A;
    WalkerState &ws = s.ws[wid];
    if (!fire_walker(s, ws, n, s.nact[wid])) return;
    const RelaxParamsDev &p = s.rp;
    double F[kFireAtoms][3], V[kFireAtoms][3];
    double m[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < kFireAtoms; ++k) {
        const int l = tid + k * kFireBlock, i = off + l;
        const bool in = l < n;
        F[k][0] = in ? b.fx[i] : 0.0;
        F[k][1] = in ? b.fy[i] : 0.0;
        F[k][2] = in ? b.fz[i] : 0.0;
        for (int c = 0; c < 3; ++c) {
            V[k][c] = in ? s.V[c * A + i] : 0.0;
            m[c] += V[k][c];
        }
    }
    const int it = ws.it, nstep0 = ws.nstep, mode = b.active[wid];
    const double dt0 = ws.dt, alpha0 = ws.alpha, E = b.out[wid].total;
    fire_sum<3>(m, sh);
    // centre-of-mass velocity removed; power, |F|^2, |V|^2, largest |F_i|^2
    double acc[3] = {0.0, 0.0, 0.0}, fm2 = 0.0;
#pragma unroll
    for (int k = 0; k < kFireAtoms; ++k) {
        if (tid + k * kFireBlock >= n) continue;
        double q = 0.0;
        for (int c = 0; c < 3; ++c) {
            V[k][c] -= m[c] / (double)n;
            acc[0] += F[k][c] * V[k][c];
            q += F[k][c] * F[k][c];
            acc[2] += V[k][c] * V[k][c];
        }
        acc[1] += q;
        fm2 = fmax(fm2, q);
    }
    for (int o = 32; o > 0; o >>= 1) fm2 = fmax(fm2, __shfl_xor(fm2, o));
    if ((tid & 63) == 0) sh[3 * kFireWaves + (tid >> 6)] = fm2;
    fire_sum<3>(acc, sh);  // its barriers cover the maxima too
    for (int k = 0; k < kFireWaves; ++k) fm2 = fmax(fm2, sh[3 * kFireWaves + k]);
    const bool conv = sqrt(acc[1]) < p.normTol || sqrt(fm2) < p.forceTol;
    const bool end = conv || it >= p.maxIter;
    double dt = dt0, alpha = alpha0;
    int nstep = nstep0;
    const bool down = acc[0] > 0.0;
    if (!end) {
        if (down) {
            if (nstep > p.N_min) {
                dt = fmin(dt * p.stepIncrease, p.maxTimeStep);
                alpha *= p.alphaDecrease;
            }
            nstep += 1;
        } else {
            nstep = 0;
            dt *= p.stepDecrease;
            alpha = p.alphaStart;
        }
        const double af = alpha0 * sqrt(acc[2]) / sqrt(acc[1]), oma = 1.0 - alpha0, fact = dt * p.timeStepUnit;
        double *px[3] = {b.x, b.y, b.z};
#pragma unroll
        for (int k = 0; k < kFireAtoms; ++k) {
            int l = tid + k * kFireBlock;
            asm volatile("" : "+v"(l));  // addresses made here, not kept across the sums
            if (l >= n) continue;
            const int i = off + l;
            for (int c = 0; c < 3; ++c) {
                double v = down ? oma * V[k][c] + af * F[k][c] : 0.0;
                const double x = s.X[c * A + i] + dt * v;
                v += fact * F[k][c];
                s.X[c * A + i] = x;
                px[c][i] = x;
                s.V[c * A + i] = v;
            }
        }
    }
    __syncthreads();  // every thread has read the walker's state
    if (tid != 0) return;
    ws.fcalls += 1;
    ws.E_last = ws.E0 = E;
    ws.fire_done = 1;  // the logic kernel that follows leaves the walker alone
    if (mode == 1) s.evals32[wid] += 1;
    if (end) {
        ws.status = conv ? 0 : 1;
        if (s.final64) {
            ws.state = ST_R_E64;
            b.active[wid] = 2;
        } else {
            ws.state = ST_DONE;  // the probe is X already
            b.active[wid] = 0;
        }
        return;
    }
    ws.it = it + 1;
    ws.dt = dt;
    ws.alpha = alpha;
    ws.nstep = nstep;
    if (down) ws.nuphill = 0;
    else ws.vf[0] = ws.vf[1] = ws.vf[2] = 0.0;
}
#endif

__global__ void __launch_bounds__(kBlock) k_search_logic(BatchDev b, SearchDev s)
{
    __shared__ double sh[4 * kBlock];
    __shared__ double lq[kLzLds];
    __shared__ WalkerState ws;
    const int wid = blockIdx.x;
    if (b.r.on && (b.zflag[wid] & AKMC_ZONE_RES)) return;  // the resident kernel advances it
    if (threadIdx.x == 0) {
        ws = s.ws[wid];
        // this step's FP32 pair kernels evaluated the walker iff it is
        // still marked FP32 here (the logic below may change the mark)
        if (b.active[wid] == 1 && !ws.fire_done) s.evals32[wid] += 1;
    }
    __syncthreads();
    if (ws.kind == WK_IDLE || ws.state == ST_DONE) return;
    const WalkerDev W = b.walkers[wid];
    if (ws.fire_done) {  // k_relax_fire has taken this micro-step
        if (threadIdx.x == 0) s.ws[wid].fire_done = 0;
        return;
    }
    Ctx C_{b, s, W.off, W.n, b.A, s.nact[wid], lq};
    // every thread keeps a private copy of the walker scalars; all threads
    // take the same branches (the scalars only change through block-wide
    // reductions), thread 0 writes them back
    WalkerState w = ws;
    walker_step(C_, w, sh);
    if (threadIdx.x == 0) s.ws[wid] = w;
}

// probes of freshly started walkers (no force call consumed yet): X for
// relax and the dimer centre.  Walkers already under way keep the probe
// their last logic step wrote (a dimer end, a Lanczos displacement).
__global__ void __launch_bounds__(kBlock) k_probe_init(BatchDev b, SearchDev s)
{
    const int wid = blockIdx.x;
    const WalkerState w = s.ws[wid];
    if (w.kind == WK_IDLE || w.state == ST_DONE || w.fcalls != 0) return;
    const WalkerDev W = b.walkers[wid];
    Ctx C_{b, s, W.off, W.n, b.A, s.nact[wid], nullptr};
    FOR_ATOMS(i) C_.probe(i, V3(s.X, 0, i), V3(s.X, 1, i), V3(s.X, 2, i));
}

#if AKMC_LOGIC_BLOCK == 256
// scatter of packed walker starts (one workgroup per walker): the free-atom
// list, the mode N of the free atoms (zero elsewhere), zero velocity,
// positions X when given, and the frozen mask, which is the complement of
// the list
__global__ void __launch_bounds__(kBlock) k_load_walkers(BatchDev b, SearchDev s, const LoadItem *items,
                                                          const double *D, const int *I)
{
    const LoadItem it = items[blockIdx.x];
    const WalkerDev W = b.walkers[it.walker];
    const int n = W.n, off = W.off, m = it.nact;
    const size_t A = b.A;
    const double *d = D + it.dbl, *x = d + 3 * (size_t)m;
    int *frozen = const_cast<int *>(s.frozen);
    int *act = const_cast<int *>(s.act);
    for (int i = threadIdx.x; i < n; i += kBlock) {
        for (int c = 0; c < 3; ++c) {
            s.N[c * A + off + i] = 0.0;
            s.V[c * A + off + i] = 0.0;
            if (it.has_x) s.X[c * A + off + i] = x[(size_t)c * n + i];
        }
        frozen[off + i] = 1;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < m; k += kBlock) {
        const int i = I[it.ints + k];  // global id
        act[off + k] = i;
        frozen[i] = 0;
        for (int c = 0; c < 3; ++c) s.N[c * A + i] = d[(size_t)c * m + k];
    }
    if (threadIdx.x == 0) const_cast<int *>(s.nact)[it.walker] = m;
}

#endif
}  // namespace

#if AKMC_LOGIC_BLOCK == 256
void akmc_launch_load_walkers(const BatchDev &b, const SearchDev &s, const LoadItem *items, int nitems,
                              const double *D, const int *I, hipStream_t st)
{
    if (nitems > 0) k_load_walkers<<<nitems, kBlock, 0, st>>>(b, s, items, D, I);
}

// the listed walkers' x, y, z slices packed walker after walker (out +
// dst[k]: x[n], y[n], z[n] of walker ws[k]); one workgroup per walker
__global__ void __launch_bounds__(kBlock) k_gather_walkers(const WalkerDev *walkers, const double *sx,
                                                           const double *sy, const double *sz, const int *ws,
                                                           const long long *dst, double *out)
{
    const WalkerDev W = walkers[ws[blockIdx.x]];
    double *o = out + dst[blockIdx.x];
    for (int a = threadIdx.x; a < W.n; a += kBlock) {
        o[a] = sx[W.off + a];
        o[W.n + a] = sy[W.off + a];
        o[2 * W.n + a] = sz[W.off + a];
    }
}

void akmc_launch_gather_walkers(const WalkerDev *walkers, const double *const src[3], const int *ws,
                                const long long *dst, int nw, double *out, hipStream_t st)
{
    if (nw > 0) k_gather_walkers<<<nw, kBlock, 0, st>>>(walkers, src[0], src[1], src[2], ws, dst, out);
}

void akmc_launch_probe_init(const BatchDev &b, const SearchDev &s, hipStream_t st)
{
    k_probe_init<<<b.W, kBlock, 0, st>>>(b, s);
}

__global__ void k_start_walkers(BatchDev b, SearchDev s, const StartItem *items, int n, int *zflag, int *harvested,
                                int *res_n)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const StartItem &it = items[k];
    s.ws[it.walker] = it.ws;
    if (zflag) zflag[it.walker] = it.zflag;
    if (harvested) harvested[it.walker] = 0;
    if (res_n) res_n[it.walker] = -1;  // the resident lists are built on its first evaluation
    b.rebuild[it.walker] = 1;
    b.active[it.walker] = it.active;
}

void akmc_launch_start_walkers(const BatchDev &b, const SearchDev &s, const StartItem *items, int nitems, int *zflag,
                               int *harvested, int *res_n, hipStream_t st)
{
    if (nitems > 0)
        k_start_walkers<<<(nitems + kBlock - 1) / kBlock, kBlock, 0, st>>>(b, s, items, nitems, zflag, harvested,
                                                                           res_n);
}

// one workgroup per walker
__global__ void __launch_bounds__(kBlock) k_harvest_pack(BatchDev b, SearchDev s, int *harvested, double *out)
{
    const int w = blockIdx.x;
    const WalkerState &ws = s.ws[w];
    if (ws.kind == WK_IDLE || ws.state != ST_DONE || harvested[w]) return;
    const WalkerDev W = b.walkers[w];
    const size_t A = b.A;
    for (int i = W.off + (int)threadIdx.x; i < W.off + W.n; i += kBlock)
        for (int c = 0; c < 3; ++c) out[(size_t)c * A + i] = s.X[(size_t)c * A + i];
    if (threadIdx.x == 0) harvested[w] = 1;
}

void akmc_launch_harvest_pack(const BatchDev &b, const SearchDev &s, int *harvested, double *out, hipStream_t st)
{
    k_harvest_pack<<<b.W, kBlock, 0, st>>>(b, s, harvested, out);
}

void akmc_launch_relax_fire(const BatchDev &b, const SearchDev &s, hipStream_t st)
{
    k_relax_fire<<<b.W, kFireBlock, 0, st>>>(b, s);
}

void akmc_launch_search_logic(const BatchDev &b, const SearchDev &s, hipStream_t st)
{
    k_search_logic<<<b.W, kBlock, 0, st>>>(b, s);
}
#else
void akmc_launch_search_logic_wide(const BatchDev &b, const SearchDev &s, hipStream_t st)
{
    k_search_logic<<<b.W, kBlock, 0, st>>>(b, s);
}
#endif
