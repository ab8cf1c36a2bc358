// Kernels of the walker state machines (search_logic.h): the logic kernel,
// walker starts, probes and harvests.
#include "search_logic.h"

namespace {

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
        if (b.active[wid] == 1) s.evals32[wid] += 1;
    }
    __syncthreads();
    if (ws.kind == WK_IDLE || ws.state == ST_DONE) return;
    const WalkerDev W = b.walkers[wid];
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
// scatter of packed walker starts (one workgroup per walker): mode N,
// zero velocity, positions X when given, the frozen mask, the free-atom
// list and its length
__global__ void __launch_bounds__(kBlock) k_load_walkers(BatchDev b, SearchDev s, const LoadItem *items,
                                                          const double *D, const int *I)
{
    const LoadItem it = items[blockIdx.x];
    const WalkerDev W = b.walkers[it.walker];
    const int n = W.n, off = W.off;
    const size_t A = b.A;
    const double *d = D + it.dbl;
    const int *iw = I + it.ints;
    int *frozen = const_cast<int *>(s.frozen);
    int *act = const_cast<int *>(s.act);
    for (int i = threadIdx.x; i < n; i += kBlock) {
        for (int c = 0; c < 3; ++c) {
            s.N[c * A + off + i] = d[(size_t)c * n + i];
            s.V[c * A + off + i] = 0.0;
            if (it.has_x) s.X[c * A + off + i] = d[(size_t)(3 + c) * n + i];
        }
        frozen[off + i] = iw[i];
    }
    for (int k = threadIdx.x; k < it.nact; k += kBlock) act[off + k] = iw[n + k];
    if (threadIdx.x == 0) const_cast<int *>(s.nact)[it.walker] = it.nact;
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
