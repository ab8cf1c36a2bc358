// Resident saddle searches on gfx950: one workgroup keeps one walker for
// several micro-steps -- evaluation and state machine alternate inside one
// launch -- instead of a chain of kernels over the whole batch per step.
//
// A search (dimer, ART, its FP64 verification, the basin-2 relax) moves only
// its free atoms.  A frozen atom's density and pair energy are a part from
// frozen neighbours, fixed for the whole search, and a part from the free
// atoms in reach.  The chain (list build, all-atom passes) evaluates a
// walker once per precision at its start and k_res_base keeps the fixed
// parts; from then on an evaluation visits
//   - the free atoms' own neighbours (densities, then forces), and
//   - per frozen atom of the zone, the free atoms in reach (a bit mask),
// about 35,000 pairs for the 75 free atoms of a 6 A region against 160,000
// for the zone's whole lists.  The energy is the sum over the zone's atoms
// plus that of the atoms outside it, which changes only with the zone.
//
// What bounds it: one walker's chain of dependent phases (lists, masks,
// reductions), with at most two workgroups of four wavefronts per CU to
// hide it.  512 walkers of 500-4000 atoms: 91 us per micro-step for
// evaluations and state machines, where the chain's kernels took 293 us; 12
// walkers: 60 us against 104 us; 128 alloy cells of 3600 atoms, searches
// with verification and basin 2: 86 us against 286 us.
//
// Results do not depend on the batch or on when the lists were built.  The
// FP32 terms summed here span fewer than 2^29 in magnitude and count, so
// their FP64 sums are exact in any order; the FP64 fixed parts are summed in
// twice the working precision.  With zones off the chain evaluates every
// atom on every step and the same kernel follows, so both modes agree bit
// for bit.
#include "search_logic.h"
#include "sc_pair.h"

namespace {

constexpr int kFree = AKMC_RES_FREE, kSlots = AKMC_RES_SLOTS, kCand = AKMC_RES_CAND;
constexpr int kBitWords = 7168;  // hit words of a list build: free atoms x candidate wavefronts
constexpr int kFreeLanes = 16;   // lanes per free atom's list
constexpr int kFreeIlp = 4;      // list entries in flight per lane
constexpr int kFzLanes = 4;      // lanes (mask words) per frozen slot
constexpr int kResSpec = 4;      // species of a resident walker's field
static_assert(kCand * sizeof(uint16_t) + kBitWords * 8 == kLzLds * sizeof(double), "the build fits the pool");
static_assert(4 * kSlots == kLzLds, "four doubles of the pool per slot");

// a resident workgroup's LDS
template <int KIND>
struct ResLds {
    double pool[kLzLds];                 // records of the zone, build scratch, Lanczos vectors
    double fx[kFree], fy[kFree], fz[kFree];  // free atoms
    uint16_t fid[kFree], fslot[kFree];   // their local indices and slots
    uint8_t zt[kSlots];                  // per slot: species, bit 7: free
    SCPairDev tab[KIND == 1 ? 1 : kResSpec * kResSpec];  // pair table (general and table kinds)
    double sh[4 * kWaves];
    int wsum[2 * kWaves];
    WalkerState ws;
};

// sqrt(x) to within half a unit in the last place or so: the hardware
// estimate and one Newton step (the general kernels' table pairs take the
// correctly rounded square root at twice the instructions)
__device__ inline float root_refined(float x)
{
    const float y = __builtin_amdgcn_rsqf(x), r = x * y;
    return __builtin_fmaf(__builtin_fmaf(-r, r, x), 0.5f * y, r);
}

// powers of U pairs: un = (a/r)^n, um = (a/r)^m, ir2 = 1/r^2.  KIND 1: one
// species pair, n = 9, m = 6; 2: a pair table with n = 9, m = 6 throughout;
// 0: any exponents (un = um = 0 for species pairs without a potential)
template <typename T, int KIND, int U>
__device__ inline void pair_terms(const double (&r2)[U], const bool (&in)[U], const SCCoef<T> &c1,
                                  const SCPairDev *const (&p)[U], T (&ir2)[U], T (&un)[U], T (&um)[U])
{
    if constexpr (KIND == 1) {
        T u2[U], rt[U];
        sc_powers_in<T, U>(r2, c1.a, ir2, u2, rt);
        pow_9_6<T, U>(u2, rt, un, um);
    } else if constexpr (KIND == 2) {
        T u2[U], rt[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const double r1[1] = {r2[u]};
            T i1[1], v1[1], t1[1];
            sc_powers_in<T, 1>(r1, sc_coef<T>(*p[u]).a, i1, v1, t1);
            ir2[u] = i1[0];
            u2[u] = v1[0];
            rt[u] = sizeof(T) == 8 ? t1[0] : T(root_refined(float(v1[0])));
            const T u4 = u2[u] * u2[u];
            un[u] = u4 * u4 * rt[u];
            um[u] = u2[u] * u4;
        }
    } else {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            ir2[u] = un[u] = um[u] = T(0);
            if (!in[u] || !p[u]->on) continue;
            const SCCoef<T> &c = sc_coef<T>(*p[u]);
            ir2[u] = recip<T>(T(r2[u]));
            const T u2 = c.a * c.a * ir2[u];
            un[u] = pow_half<T>(u2, p[u]->n_int, c.n);
            um[u] = pow_half<T>(u2, p[u]->m_int, c.m);
        }
    }
}

template <typename T, int KIND>
__device__ inline const SCCoef<T> &coef_of(const SCCoef<T> &c1, const SCPairDev *p)
{
    if constexpr (KIND == 1) return c1;
    else return sc_coef<T>(*p);
}

// density and half pair energy of atom i from U partners, added in order
template <typename T, int KIND, int U>
__device__ inline void add_density(const WalkerDev &W, double rc2, const SCCoef<T> &c1, const SCPairDev *const (&p)[U],
                                   double xi, double yi, double zi, const double (&px)[U], const double (&py)[U],
                                   const double (&pz)[U], const bool (&ok)[U], double &rho, double &ep)
{
    double r2[U];
    bool in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        double dx = xi - px[u], dy = yi - py[u], dz = zi - pz[u];
        min_image(dx, dy, dz, W);
        r2[u] = dx * dx + dy * dy + dz * dz;
        in[u] = ok[u] && r2[u] <= rc2 && r2[u] > 1.0e-16;
    }
    T ir2[U], un[U], um[U];
    pair_terms<T, KIND, U>(r2, in, c1, p, ir2, un, um);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const SCCoef<T> &c = coef_of<T, KIND>(c1, p[u]);
        T eh = in[u] ? T(0.5) * c.eps * un[u] : T(0);
        T rh = in[u] ? c.rho_coef * um[u] : T(0);
        if constexpr (sizeof(T) == 4) {
            asm("" : "+v"(eh));
            asm("" : "+v"(rh));
        }
        ep += double(eh);
        rho += double(rh);
    }
}

// 1/sqrt(rho) for the force pass (-1: no density)
template <typename T>
__device__ inline T inv_root(double rho)
{
    return rho < 1.0e-8 ? T(-1) : T(1.0 / sqrt(rho));
}

// exclusive prefix over the workgroup of a flag, in thread order; total gets
// the sum.  slot alternates between two scratch rows, so one barrier does.
__device__ inline int flag_prefix(bool v, int *wsum, int row, int &total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long bal = __ballot(v);
    if (lane == 0) wsum[row * kWaves + wave] = __popcll(bal);
    __syncthreads();
    int before = 0, all = 0;
    for (int k = 0; k < kWaves; ++k) {
        const int t = wsum[row * kWaves + k];
        if (k < wave) before += t;
        all += t;
    }
    total = all;
    return before + __popcll(bal & ((1ull << lane) - 1ull));
}

// The lists of a resident walker from its free atoms' positions (in LDS):
// the zone (the free atoms and every frozen atom within rc + skin/2 of one:
// between builds a free atom moves at most skin/2 and a frozen one not at
// all), the masks of its frozen atoms and the free atoms' neighbours (free
// ones within rc + skin), all in ascending index order.  Candidates are the
// atoms within rc + skin of the free atoms' box.  false: past a capacity.
template <int KIND>
__device__ __forceinline__ bool res_build(const BatchDev &b, const SearchDev &s, const WalkerDev &W, ResLds<KIND> &L,
                                          int nf)
{
    const int w = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const ResidentDev &R = b.r;
    uint16_t *cand = reinterpret_cast<uint16_t *>(L.pool);
    unsigned long long *bits = reinterpret_cast<unsigned long long *>(L.pool + kCand / 4);
    const double rl2 = b.field->rlist2, rz2 = b.field->rzone2;
    // the free atoms' box: an arc of the cell per axis around the first one
    double lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
    const double o[3] = {L.fx[0], L.fy[0], L.fz[0]};
    for (int f = tid; f < nf; f += kBlock) {
        double d[3] = {L.fx[f] - o[0], L.fy[f] - o[1], L.fz[f] - o[2]};
        min_image(d[0], d[1], d[2], W);
        for (int c = 0; c < 3; ++c) {
            lo[c] = fmin(lo[c], d[c]);
            hi[c] = fmax(hi[c], d[c]);
        }
    }
    double bc[3], bh[3];
    for (int c = 0; c < 3; ++c) {
        const double h = bmax(hi[c], L.sh), l = -bmax(-lo[c], L.sh);
        bc[c] = o[c] + 0.5 * (l + h);
        bh[c] = 0.5 * (h - l);
    }
    int nc = 0, row = 0;
    for (int c0 = 0; c0 < W.n; c0 += kBlock, row ^= 1) {
        const int j = c0 + tid;
        bool keep = false;
        if (j < W.n) {
            const int i = W.off + j;
            double dx = b.x[i] - bc[0], dy = b.y[i] - bc[1], dz = b.z[i] - bc[2];
            min_image(dx, dy, dz, W);
            const double ex = fmax(fabs(dx) - bh[0], 0.0), ey = fmax(fabs(dy) - bh[1], 0.0),
                         ez = fmax(fabs(dz) - bh[2], 0.0);
            keep = ex * ex + ey * ey + ez * ez <= rl2 * (1.0 + 1.0e-9);
            b.zmark[i] = 0;
        }
        int tot;
        const int at = nc + flag_prefix(keep, L.wsum, row, tot);
        if (keep && at < kCand) cand[at] = uint16_t(j);
        nc += tot;
    }
    const int ncw = (nc + 63) / 64;
    __syncthreads();
    if (nc > kCand || nf * ncw > kBitWords) return false;
    // every candidate against every free atom: its mask (frozen candidates)
    // and, by ballot, the free atoms' hit words over the candidates
    int nz = 0, nfree = 0;
    for (int c0 = 0; c0 < nc; c0 += kBlock) {
        const int c = c0 + tid;
        const bool has = c < nc;
        const int j = has ? cand[c] : 0, i = W.off + j;
        const double x = b.x[i], y = b.y[i], z = b.z[i];
        const bool fr = s.frozen[i] != 0;
        const double lim = fr ? rz2 : rl2;
        unsigned long long m[kFzLanes] = {};
        const int word = (c0 >> 6) + wave;
        for (int f0 = 0; f0 < nf; f0 += kFzLanes) {
#pragma unroll
            for (int q = 0; q < kFzLanes; ++q) {
                const int f = f0 + q < nf ? f0 + q : 0;
                double dx = x - L.fx[f], dy = y - L.fy[f], dz = z - L.fz[f];
                min_image(dx, dy, dz, W);
                const bool hit = has && f0 + q < nf && dx * dx + dy * dy + dz * dz <= lim && L.fid[f] != j;
                const unsigned long long bal = __ballot(hit);
                if (lane == 0 && word < ncw && f0 + q < nf) bits[f * ncw + word] = bal;
                m[q] |= (unsigned long long)hit << (f0 >> 2);
            }
        }
        const bool member = has && (!fr || (m[0] | m[1] | m[2] | m[3]) != 0ull);
        int tot, totf;
        const int sl = nz + flag_prefix(member, L.wsum, 0, tot);
        const int fi = nfree + flag_prefix(has && !fr, L.wsum, 1, totf);
        if (has) cand[c] = member ? uint16_t(sl) : uint16_t(0xFFFF);
        if (member && sl < kSlots) {
            R.slot[(size_t)w * kSlots + sl] = uint16_t(j);
            unsigned long long *mk = R.mask + ((size_t)w * kSlots + sl) * kFzLanes;
            for (int q = 0; q < kFzLanes; ++q) mk[q] = fr ? m[q] : 0ull;
            if (!fr) {
                L.fslot[fi] = uint16_t(sl);
                R.fslot[w * kFree + fi] = uint16_t(sl);
            }
            b.zmark[i] = 1;
        }
        nz += tot;
        nfree += totf;
        __syncthreads();  // the next round reuses the scratch rows
    }
    if (nz > kSlots) return false;
    // the free atoms' lists from their hit words, one (atom, word) per thread
    for (int t = tid; t < nf * ncw; t += kBlock) {
        const int f = t / ncw, wd = t - f * ncw;
        const unsigned long long *bw = bits + f * ncw;
        int at = 0;
        for (int v = 0; v < wd; ++v) at += __popcll(bw[v]);
        uint16_t *fl = R.flist + ((size_t)w * kFree + f) * R.fcap;
        for (unsigned long long m = bw[wd]; m; m &= m - 1ull, ++at)
            if (at < R.fcap) fl[at] = cand[64 * wd + __ffsll((long long)m) - 1];
        if (wd == ncw - 1) {
            R.fcnt[w * kFree + f] = at < R.fcap ? at : R.fcap;
            if (at > R.fcap) atomicOr(b.overflow, AKMC_OV_LIST);
        }
    }
    for (int f = tid; f < nf; f += kBlock) {
        R.ref[((size_t)w * 3 + 0) * kFree + f] = L.fx[f];
        R.ref[((size_t)w * 3 + 1) * kFree + f] = L.fy[f];
        R.ref[((size_t)w * 3 + 2) * kFree + f] = L.fz[f];
    }
    if (tid == 0) {
        R.n[w] = nz;
        R.eok[w] = 0;
        b.nz[w] = nz;
        atomicAdd(b.rebuild_count, 1ull);
    }
    __syncthreads();
    return true;
}

// energies of the atoms outside the zone (fixed parts only: no free atom is
// in their reach), in index order per thread
template <int KIND>
__device__ __forceinline__ void res_outside(const BatchDev &b, const WalkerDev &W, ResLds<KIND> &L, int nz, int prec)
{
    const int w = blockIdx.x, tid = threadIdx.x;
    uint32_t *in = reinterpret_cast<uint32_t *>(L.pool);
    for (int k = tid; k < (AKMC_RES_ATOMS + 32) / 32; k += kBlock) in[k] = 0u;
    __syncthreads();
    for (int k = tid; k < nz; k += kBlock) {
        const int j = b.r.slot[(size_t)w * kSlots + k];
        atomicOr(&in[j >> 5], 1u << (j & 31));
    }
    __syncthreads();
    double v[2] = {0.0, 0.0};
    for (int j = tid; j < W.n; j += kBlock) {
        if ((in[j >> 5] >> (j & 31)) & 1u) continue;
        v[0] -= sqrt(b.r.base_rho[prec][W.off + j]);
        v[1] += b.r.base_ep[prec][W.off + j];
    }
    bsum<2>(v, L.sh);
    if (tid == 0) {
        double *e = b.r.eout + ((size_t)w * 2 + prec) * 2;
        e[0] = v[0];
        e[1] = v[1];
        b.r.eok[w] |= 1 << prec;
    }
    __syncthreads();
}

// one evaluation at the free positions in LDS: forces of the free atoms and
// the walker's energy record
template <typename T, int KIND>
__device__ __forceinline__ void res_eval(const BatchDev &b, const WalkerDev &W, ResLds<KIND> &L, int nf, int nz)
{
    constexpr int prec = sizeof(T) == 8 ? 1 : 0;
    const int w = blockIdx.x, tid = threadIdx.x;
    const FieldDev &F = *b.field;
    const SCCoef<T> c1 = sc_coef<T>(F.sc[0]);
    const double rc2 = F.rc2;
    const int ns = F.nspec;
    const ResidentDev &R = b.r;
    const double *rx = L.pool, *ry = rx + kSlots, *rz = ry + kSlots;
    T *rw = reinterpret_cast<T *>(L.pool + 3 * kSlots);  // 1/sqrt(rho) per slot
    double many = 0.0, pair = 0.0;
    // frozen slots: four lanes each, one mask word per lane, two of its free
    // atoms at a time; the next slot's loads go out before this one's pairs
    const unsigned long long *mask = R.mask + (size_t)w * kSlots * kFzLanes;
    const uint16_t *slot = R.slot + (size_t)w * kSlots;
    {
        int t = tid;
        unsigned long long mn = t < kFzLanes * nz ? mask[t] : 0ull;
        int jn = t < kFzLanes * nz ? slot[t / kFzLanes] : 0;
        for (; t < kFzLanes * nz; t += kBlock) {
            unsigned long long m = mn;
            const int i = W.off + jn, sl = t / kFzLanes, q = t % kFzLanes;
            const double brho = R.base_rho[prec][i], bep = R.base_ep[prec][i];
            if (t + kBlock < kFzLanes * nz) {
                mn = mask[t + kBlock];
                jn = slot[(t + kBlock) / kFzLanes];
            }
            const int zt = L.zt[sl];
            if (zt & 128) continue;  // a free slot (all four lanes)
            const double xi = rx[sl], yi = ry[sl], zi = rz[sl];
            double rho = 0.0, ep = 0.0;
            while (m) {
                double px[2], py[2], pz[2];
                bool ok[2];
                const SCPairDev *p[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    ok[u] = m != 0ull;
                    const int f = ok[u] ? kFzLanes * (__ffsll((long long)m) - 1) + q : 0;
                    m &= m - 1ull;
                    px[u] = L.fx[f];
                    py[u] = L.fy[f];
                    pz[u] = L.fz[f];
                    p[u] = KIND == 1 ? nullptr : L.tab + (zt & 127) * ns + (L.zt[L.fslot[f]] & 127);
                }
                add_density<T, KIND, 2>(W, rc2, c1, p, xi, yi, zi, px, py, pz, ok, rho, ep);
            }
            rho = lane_group_sum<kFzLanes>(rho) + brho;
            ep = lane_group_sum<kFzLanes>(ep) + bep;
            if (q == 0) {
                rw[sl] = inv_root<T>(rho);
                many -= sqrt(rho);
                pair += ep;
            }
        }
    }
    // free atoms: kFreeLanes lanes per list, entries strided over the lanes,
    // the next batch (of this atom or the next) in flight during a batch
    const int g = tid / kFreeLanes, sub = tid % kFreeLanes;
    constexpr int kGroups = kBlock / kFreeLanes, kBatch = kFreeLanes * kFreeIlp;
    const int *fcnt = R.fcnt + w * kFree;
    const uint16_t *flist = R.flist + (size_t)w * kFree * R.fcap;
    auto fetch = [&](int f, int k, int cnt, int (&e)[kFreeIlp]) {
#pragma unroll
        for (int u = 0; u < kFreeIlp; ++u) {
            const int kk = k + u * kFreeLanes;
            e[u] = kk < cnt ? int(flist[(size_t)f * R.fcap + kk]) : -1;
        }
    };
    {
        int f = g, cnt = f < nf ? fcnt[f] : 0, en[kFreeIlp];
        if (f < nf) fetch(f, sub, cnt, en);
        while (f < nf) {
            const int fn = f + kGroups, cn = fn < nf ? fcnt[fn] : 0;
            const int sl = L.fslot[f], zt = L.zt[sl] & 127;
            const double xi = L.fx[f], yi = L.fy[f], zi = L.fz[f];
            double rho = 0.0, ep = 0.0;
            for (int k = sub; k < cnt || k == sub; k += kBatch) {
                int e[kFreeIlp];
#pragma unroll
                for (int u = 0; u < kFreeIlp; ++u) e[u] = en[u];
                if (k + kBatch < cnt) fetch(f, k + kBatch, cnt, en);
                else if (fn < nf) fetch(fn, sub, cn, en);
                double px[kFreeIlp], py[kFreeIlp], pz[kFreeIlp];
                bool ok[kFreeIlp];
                const SCPairDev *p[kFreeIlp];
#pragma unroll
                for (int u = 0; u < kFreeIlp; ++u) {
                    ok[u] = e[u] >= 0;
                    const int j = ok[u] ? e[u] : sl;
                    px[u] = rx[j];
                    py[u] = ry[j];
                    pz[u] = rz[j];
                    p[u] = KIND == 1 ? nullptr : L.tab + zt * ns + (L.zt[j] & 127);
                }
                add_density<T, KIND, kFreeIlp>(W, rc2, c1, p, xi, yi, zi, px, py, pz, ok, rho, ep);
            }
            rho = lane_group_sum<kFreeLanes>(rho);
            ep = lane_group_sum<kFreeLanes>(ep);
            if (sub == 0) {
                rw[sl] = inv_root<T>(rho);
                many -= sqrt(rho);
                pair += ep;
            }
            f = fn;
            cnt = cn;
        }
    }
    __syncthreads();
    // forces of the free atoms (the expressions of the chain's pass 2)
    {
        int f = g, cnt = f < nf ? fcnt[f] : 0, en[kFreeIlp];
        if (f < nf) fetch(f, sub, cnt, en);
        while (f < nf) {
            const int fn = f + kGroups, cn = fn < nf ? fcnt[fn] : 0;
            const int sl = L.fslot[f], zt = L.zt[sl] & 127;
            const double xi = L.fx[f], yi = L.fy[f], zi = L.fz[f];
            const T isi = rw[sl];
            double fx = 0.0, fy = 0.0, fz = 0.0;
            for (int k = sub; k < cnt || k == sub; k += kBatch) {
                int e[kFreeIlp];
#pragma unroll
                for (int u = 0; u < kFreeIlp; ++u) e[u] = en[u];
                if (k + kBatch < cnt) fetch(f, k + kBatch, cnt, en);
                else if (fn < nf) fetch(fn, sub, cn, en);
                double dx[kFreeIlp], dy[kFreeIlp], dz[kFreeIlp], r2[kFreeIlp];
                T isj[kFreeIlp];
                bool in[kFreeIlp];
                const SCPairDev *p[kFreeIlp];
#pragma unroll
                for (int u = 0; u < kFreeIlp; ++u) {
                    const int j = e[u] >= 0 ? e[u] : sl;
                    dx[u] = xi - rx[j];
                    dy[u] = yi - ry[j];
                    dz[u] = zi - rz[j];
                    isj[u] = rw[j];
                    p[u] = KIND == 1 ? nullptr : L.tab + zt * ns + (L.zt[j] & 127);
                    min_image(dx[u], dy[u], dz[u], W);
                    r2[u] = dx[u] * dx[u] + dy[u] * dy[u] + dz[u] * dz[u];
                    in[u] = e[u] >= 0 && r2[u] <= rc2 && r2[u] > 1.0e-16;
                }
                T ir2[kFreeIlp], un[kFreeIlp], um[kFreeIlp];
                pair_terms<T, KIND, kFreeIlp>(r2, in, c1, p, ir2, un, um);
#pragma unroll
                for (int u = 0; u < kFreeIlp; ++u) {
                    const SCCoef<T> &c = coef_of<T, KIND>(c1, p[u]);
                    const T fs = c.fs_coef * un[u];
                    const T fm = (isi >= T(0) && isj[u] >= T(0)) ? c.fm_coef * (isi + isj[u]) * um[u] : T(0);
                    T ft = in[u] ? (fs - fm) * ir2[u] : T(0);
                    if constexpr (sizeof(T) == 4) asm("" : "+v"(ft));
                    const double dft = double(ft);
                    fx += dft * dx[u];
                    fy += dft * dy[u];
                    fz += dft * dz[u];
                }
            }
            fx = lane_group_sum<kFreeLanes>(fx);
            fy = lane_group_sum<kFreeLanes>(fy);
            fz = lane_group_sum<kFreeLanes>(fz);
            if (sub == 0) {
                const int i = W.off + L.fid[f];
                b.fx[i] = fx;
                b.fy[i] = fy;
                b.fz[i] = fz;
            }
            f = fn;
            cnt = cn;
        }
    }
    double v[2] = {many, pair};
    bsum<2>(v, L.sh);
    if (tid == 0) {
        const double *e = R.eout + ((size_t)w * 2 + prec) * 2;
        WalkerOut o;
        o.many = e[0] + v[0];
        o.vdw = e[1] + v[1];
        o.real = o.rcp = o.self = 0.0;
        o.total = o.many + o.vdw;
        for (int c = 0; c < 6; ++c) o.stress[c] = 0.0;
        b.out[w] = o;
    }
    __syncthreads();
}

// Micro-steps of resident walkers, one workgroup each.  A walker whose full
// evaluation in its precision is pending has had it from the chain that ran
// before this launch when the launch begins; one that comes to need it later
// (a search entering FP64 verification) waits for the next launch.
template <int KIND>
__global__ void __launch_bounds__(kBlock, 2) k_search_resident(BatchDev b, SearchDev s, int nsteps, int logic)
{
    __shared__ ResLds<KIND> L;
    const int wid = blockIdx.x, tid = threadIdx.x;
    int flags = b.zflag[wid];
    if (!(flags & AKMC_ZONE_RES) || b.active[wid] == 0) return;
    if (tid == 0) L.ws = s.ws[wid];
    if constexpr (KIND != 1) stage_sc_table(*b.field, L.tab);
    __syncthreads();
    if (L.ws.kind == WK_IDLE || L.ws.state == ST_DONE) return;
    const WalkerDev W = b.walkers[wid];
    const int nf = s.nact[wid];
    Ctx C_{b, s, W.off, W.n, b.A, nf, L.pool};
    const double h2 = b.field->half_skin2;
    int nz = b.r.n[wid], evals32 = 0;
    if (nz >= 0)
        for (int f = tid; f < nf; f += kBlock) L.fslot[f] = b.r.fslot[wid * kFree + f];
    for (int f = tid; f < nf; f += kBlock) L.fid[f] = uint16_t(s.act[W.off + f] - W.off);
    bool loaded = false, too_big = false;  // loaded: the zone's records are in the pool
    for (int step = 0; step < nsteps; ++step) {
        __syncthreads();
        if (L.ws.state == ST_DONE) break;
        const int mode = b.active[wid], prec = mode == 2 ? 1 : 0;
        const int full = prec ? AKMC_ZONE_FULL64 : AKMC_ZONE_FULL32;
        if (flags & full) {
            if (step > 0) break;
            flags &= ~full;
            if (tid == 0) b.r.eok[wid] &= ~(1 << prec);
        }
        bool moved = nz < 0;
        for (int f = tid; f < nf; f += kBlock) {
            const int i = W.off + L.fid[f];
            const double x = b.x[i], y = b.y[i], z = b.z[i];
            L.fx[f] = x;
            L.fy[f] = y;
            L.fz[f] = z;
            if (nz >= 0) {
                const double *r = b.r.ref + (size_t)wid * 3 * kFree + f;
                const double dx = x - r[0], dy = y - r[kFree], dz = z - r[2 * kFree];
                moved |= dx * dx + dy * dy + dz * dz > h2;
            }
        }
        if (__syncthreads_or(moved)) {
            if (!res_build(b, s, W, L, nf)) {
                too_big = true;
                break;
            }
            nz = b.r.n[wid];
            loaded = false;
        }
        if (!(b.r.eok[wid] & (1 << prec))) {
            res_outside(b, W, L, nz, prec);
            loaded = false;
        }
        if (!loaded) {
            for (int k = tid; k < nz; k += kBlock) {
                const int i = W.off + b.r.slot[(size_t)wid * kSlots + k];
                L.pool[k] = b.x[i];
                L.pool[kSlots + k] = b.y[i];
                L.pool[2 * kSlots + k] = b.z[i];
                L.zt[k] = uint8_t(b.type[i] | (s.frozen[i] ? 0 : 128));
            }
            loaded = true;
        } else {
            for (int f = tid; f < nf; f += kBlock) {
                const int k = L.fslot[f];
                L.pool[k] = L.fx[f];
                L.pool[kSlots + k] = L.fy[f];
                L.pool[2 * kSlots + k] = L.fz[f];
            }
        }
        __syncthreads();
        if (prec) res_eval<double, KIND>(b, W, L, nf, nz);
        else res_eval<float, KIND>(b, W, L, nf, nz);
        if (!logic) break;
        evals32 += mode == 1;
        // the walker's scalars are private to each thread during its step (all
        // threads take the same branches) and in LDS during the evaluations
        WalkerState w = L.ws;
        if (w.kind == WK_VERIFY) loaded = false;  // its Lanczos vectors take the pool
        walker_step(C_, w, L.sh);
        __syncthreads();
        if (tid == 0) L.ws = w;
    }
    __syncthreads();
    if (tid == 0) {
        b.zflag[wid] = flags;
        if (too_big) L.ws.too_big = 1;
        if (logic || too_big) s.ws[wid] = L.ws;
        s.evals32[wid] += evals32;
    }
}

// a sum kept in twice the working precision (Knuth's two-sum)
struct Sum2 {
    double h, l;
    __device__ inline void add(double v)
    {
        const double t = __dadd_rn(h, v), z = __dsub_rn(t, h);
        l = __dadd_rn(l, __dadd_rn(__dsub_rn(h, __dsub_rn(t, z)), __dsub_rn(v, z)));
        h = t;
    }
};

constexpr int kBaseLanes = 4, kBaseSplit = 16, kBaseBlock = 256;

template <typename T, int KIND>
__device__ inline void res_base_atoms(const BatchDev &b, const WalkerDev &W, const SCPairDev *tab)
{
    constexpr int prec = sizeof(T) == 8 ? 1 : 0;
    const FieldDev &F = *b.field;
    const SCCoef<T> c1 = sc_coef<T>(F.sc[0]);
    const int sub = threadIdx.x % kBaseLanes;
    constexpr int per = kBaseBlock / kBaseLanes;
    for (int l = blockIdx.y * per + (int)threadIdx.x / kBaseLanes; l < W.n; l += kBaseSplit * per) {
        const int i = W.off + l, cnt = b.nnb[i];
        const double xi = b.x[i], yi = b.y[i], zi = b.z[i];
        Sum2 rho{0.0, 0.0}, ep{0.0, 0.0};
        for (int k = sub; k < cnt; k += kBaseLanes) {
            const int j = W.off + int(nbr_entry(b, k, i) & AKMC_NB_JMASK);
            const bool ok[1] = {b.zfrozen[j] != 0};
            const double px[1] = {b.x[j]}, py[1] = {b.y[j]}, pz[1] = {b.z[j]};
            const SCPairDev *p[1] = {KIND == 1 ? nullptr : tab + b.type[i] * F.nspec + b.type[j]};
            double r = 0.0, e = 0.0;
            add_density<T, KIND, 1>(W, F.rc2, c1, p, xi, yi, zi, px, py, pz, ok, r, e);
            rho.add(r);
            ep.add(e);
        }
        for (int o = kBaseLanes / 2; o > 0; o >>= 1) {
            const double rh = __shfl_xor(rho.h, o), rl = __shfl_xor(rho.l, o);
            const double eh = __shfl_xor(ep.h, o), el = __shfl_xor(ep.l, o);
            rho.add(rh);
            rho.l += rl;
            ep.add(eh);
            ep.l += el;
        }
        if (sub == 0) {
            b.r.base_rho[prec][i] = rho.h + rho.l;
            b.r.base_ep[prec][i] = ep.h + ep.l;
        }
    }
}

// The parts of every atom's density and pair energy that come from frozen
// neighbours, for the resident walkers the chain evaluates on this step
// (once per search and precision; kBaseSplit workgroups per walker)
template <int KIND>
__global__ void __launch_bounds__(kBaseBlock) k_res_base(BatchDev b)
{
    __shared__ SCPairDev tab[KIND == 1 ? 1 : kResSpec * kResSpec];
    const int w = blockIdx.x, mode = b.active[w], f = b.zflag[w];
    if (mode == 0 || !(f & AKMC_ZONE_RES)) return;
    if (!b.zone_off && !(f & (mode == 2 ? AKMC_ZONE_FULL64 : AKMC_ZONE_FULL32))) return;
    if constexpr (KIND != 1) stage_sc_table(*b.field, tab);
    const WalkerDev W = b.walkers[w];
    if (mode == 2) res_base_atoms<double, KIND>(b, W, tab);
    else res_base_atoms<float, KIND>(b, W, tab);
}

__global__ void k_leave_resident(BatchDev b)
{
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= b.W || !(b.zflag[w] & AKMC_ZONE_RES)) return;
    b.zflag[w] = AKMC_ZONE_ON | AKMC_ZONE_FULL32 | AKMC_ZONE_FULL64 | AKMC_ZONE_RESET;
    b.rebuild[w] = 1;
}

}  // namespace

void akmc_launch_res_base(const BatchDev &b, const FieldDev &hf, hipStream_t st)
{
    const dim3 g(b.W, kBaseSplit);
    switch (akmc_sc_kind(hf)) {
    case 1: k_res_base<1><<<g, kBaseBlock, 0, st>>>(b); break;
    case 2: k_res_base<2><<<g, kBaseBlock, 0, st>>>(b); break;
    default: k_res_base<0><<<g, kBaseBlock, 0, st>>>(b);
    }
}

void akmc_launch_search_resident(const BatchDev &b, const FieldDev &hf, const SearchDev &s, int nsteps, int logic,
                                 hipStream_t st)
{
    switch (akmc_sc_kind(hf)) {
    case 1: k_search_resident<1><<<b.W, kBlock, 0, st>>>(b, s, nsteps, logic); break;
    case 2: k_search_resident<2><<<b.W, kBlock, 0, st>>>(b, s, nsteps, logic); break;
    default: k_search_resident<0><<<b.W, kBlock, 0, st>>>(b, s, nsteps, logic);
    }
}

void akmc_launch_leave_resident(const BatchDev &b, hipStream_t st)
{
    k_leave_resident<<<(b.W + 255) / 256, 256, 0, st>>>(b);
}
