// Resident saddle searches on gfx950: one workgroup keeps one walker for
// several micro-steps -- evaluation and state machine alternate inside one
// launch -- instead of a chain of kernels over the whole batch per step.
//
// A search (dimer, ART, its FP64 verification, the basin-2 relax) moves only
// its free atoms.  A frozen atom's density and pair energy are a part from
// frozen neighbours, fixed for the whole search, and a part from the free
// atoms in reach.  The chain (list build, all-atom passes) evaluates a
// walker once, on its first micro-step, and k_res_base keeps the fixed parts
// in the precisions it may come to; from then on an evaluation visits
//   - the free atoms' own neighbours (densities, then forces), and
//   - per frozen atom of the zone, the free atoms in reach (a bit mask),
// about 35,000 pairs for the 75 free atoms of a 6 A region against 160,000
// for the zone's whole lists.  The energy is the sum over the zone's atoms
// plus that of the atoms outside it, which changes only with the zone.
//
// What bounds it: one walker's chain of dependent phases (gathers, pair
// terms, sums, the state machine's reductions; one walker alone runs at 76%
// of the rate of two on a CU), so a workgroup has eight wavefronts, two fit
// a CU, the functions are out of line for 128 registers each, lists and
// records are in LDS, and sums go by DPP moves.  512 walkers of 500-4000
// atoms: 65 us per micro-step for evaluations and state machines, where the
// chain's kernels took 293 us (91 us with four wavefronts and lists in
// global memory); 12 walkers: 37 us against 104 us.
//
// A walker's results do not depend on its batch: whether it is resident, when
// its lists are built and every order of summation follow from the walker
// alone.  The terms are the chain's, in another order: FP32 density and energy
// terms span less than 2^29 in magnitude and count at any distance a search
// meets, so their FP64 sums are the chain's bit for bit; force sums (products
// with FP64 displacements) and FP64 sums differ in their last bits, and a list
// built elsewhere along the way would change them too.  The FP64 fixed parts
// are summed in twice the working precision.  With zones off the chain
// evaluates every atom on every step and this kernel still advances the
// walker, so both modes agree bit for bit.
#define AKMC_LOGIC_BLOCK 512
#include "search_logic.h"
#include "sc_pair.h"

namespace {

constexpr int kFree = AKMC_RES_FREE, kSlots = AKMC_RES_SLOTS, kCand = AKMC_RES_CAND;
constexpr int kBitWords = 6784;  // hit words of a list build's strip: free atoms x candidate wavefronts
constexpr int kFreeLanes = 16;   // lanes per free atom's list
constexpr int kFreeIlp = 5;      // list entries in flight per lane: two batches for a bulk list of 155
constexpr int kFreeIlp64 = 2;    // FP64 entries: five spill 356 bytes of registers (alloy searches 33.3 -> 29.6 ms)
constexpr int kFzLanes = 4;      // lanes (mask words) per frozen slot
constexpr int kFzIlp = 2;        // free atoms of a mask word in flight per lane
constexpr int kClass = 8;        // frozen slots are served in classes of similar reach
constexpr int kResSpec = 4;      // species of a resident walker's field
static_assert(kCand * sizeof(uint16_t) + kBitWords * 8 + 3 * kFree * sizeof(float) == kLzLds * sizeof(double),
              "the build fits the pool");
static_assert(4 * kSlots == kLzLds, "four doubles of the pool per slot");

// a resident workgroup's LDS
template <int KIND>
struct ResLds {
    double pool[kLzLds];                 // records of the zone, build scratch, Lanczos vectors
    double fx[kFree], fy[kFree], fz[kFree];  // free atoms
    int fofs[kFree + 1];                 // start of each free atom's list among all of them
    uint16_t fid[kFree], fslot[kFree];   // their local indices and slots
    uint8_t zt[kSlots];                  // per slot: species
    SCPairDev tab[KIND == 1 ? 1 : kResSpec * kResSpec];  // pair table (general and table kinds)
    double sh[4 * kWaves];
    int wsum[2 * kWaves];
    WalkerState ws;
};

// the workgroup's LDS; one variable, so that the functions below, kept out
// of line for their own register allocations, address it directly
template <int KIND>
__device__ __forceinline__ ResLds<KIND> &res_lds()
{
    __shared__ ResLds<KIND> L;
    return L;
}

// an object every thread of the wavefront reads at one address, through
// scalar loads (it does not change while the kernel runs)
template <typename T>
__device__ __forceinline__ T load_uniform(const T *p)
{
    const unsigned long long v = reinterpret_cast<unsigned long long>(p);
    const unsigned lo = __builtin_amdgcn_readfirstlane(unsigned(v)), hi = __builtin_amdgcn_readfirstlane(unsigned(v >> 32));
    typedef const __attribute__((address_space(4))) T CT;
    T out;
    __builtin_memcpy(&out, (CT *)((unsigned long long)hi << 32 | lo), sizeof(T));
    return out;
}

// v of the lane that CTRL (a DPP row operation) pairs this one with
template <int CTRL>
__device__ __forceinline__ double dpp_of(double v)
{
    const long long w = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, int(w), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, int(w >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double((long long)(unsigned)lo | (long long)hi << 32);
}

// sum over the LPA (4 or 16) consecutive lanes of a group, the same bits on
// all of them: neighbours, pairs (quad permutes), quads and halves of a row
// (mirrors); register moves instead of the LDS shuffles of lane_group_sum
template <int LPA>
__device__ __forceinline__ double row_sum(double v)
{
    static_assert(LPA == 4 || LPA == 16, "quads or rows");
    v += dpp_of<0xB1>(v);  // quad_perm [1,0,3,2]
    v += dpp_of<0x4E>(v);  // quad_perm [2,3,0,1]
    if constexpr (LPA == 16) {
        v += dpp_of<0x141>(v);  // row_half_mirror
        v += dpp_of<0x140>(v);  // row_mirror
    }
    return v;
}

// During evaluations the pool holds x, y, z and 1/sqrt(rho) per zone slot,
// S doubles each, then the free atoms' lists when they fit (75 free atoms:
// 28 KB and 24 KB of the 64 KB)
__device__ inline int slot_stride(int nz) { return (nz + 15) & ~15; }
__device__ inline bool lists_fit(int entries, int S) { return entries <= 4 * (kLzLds - 4 * S); }

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
#pragma unroll
        for (int u = 0; u < U; ++u) table_9_6<T>(r2[u], sc_coef<T>(*p[u]), ir2[u], un[u], um[u]);
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
__device__ __attribute__((noinline)) bool res_build(const ResArgs *args, int nf)
{
    ResLds<KIND> &L = res_lds<KIND>();
    const BatchDev b = load_uniform(&args->b);
    const SearchDev s = load_uniform(&args->s);
    const WalkerDev W = load_uniform(b.walkers + blockIdx.x);
    const int w = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const ResidentDev &R = b.r;
    uint16_t *cand = reinterpret_cast<uint16_t *>(L.pool);
    unsigned long long *bits = reinterpret_cast<unsigned long long *>(L.pool + kCand / 4);
    float *gx = reinterpret_cast<float *>(bits + kBitWords), *gy = gx + kFree, *gz = gy + kFree;  // from the box centre
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
    if (nc > kCand) return false;
    // the hit words of this many free atoms fit at a time (106 with every
    // candidate's worth; a 6 A region's 75 atoms always)
    const int strip = min(nf, (kBitWords / ncw) & ~(kFzLanes - 1));
    // every candidate against every free atom: its mask (frozen candidates)
    // and, by ballot, the free atoms' hit words over the candidates.  FP32
    // distances with a margin above their rounding (coordinates of up to L/2,
    // 2^-24 of that each, so 2 r sqrt(3) L 2^-24 = 2e-7 r L on a square): an
    // entry past its radius adds nothing, the evaluation tests every pair in
    // FP64
    for (int f = tid; f < nf; f += kBlock) {
        double dx = L.fx[f] - bc[0], dy = L.fy[f] - bc[1], dz = L.fz[f] - bc[2];
        min_image(dx, dy, dz, W);
        gx[f] = float(dx);
        gy[f] = float(dy);
        gz[f] = float(dz);
    }
    __syncthreads();
    const float L0 = float(W.L[0]), L1 = float(W.L[1]), L2 = float(W.L[2]);
    const float i0 = float(W.invL[0]), i1 = float(W.invL[1]), i2 = float(W.invL[2]);
    const float margin = 1.0e-6f * float(sqrt(rl2)) * fmaxf(fmaxf(L0, L1), fmaxf(L2, 16.0f));
    // atom j of the walker in the box's frame, and whether free atom f is
    // within its radius
    auto place = [&](int j, float &x, float &y, float &z, float &lim) {
        const int i = W.off + j;
        double xd = b.x[i] - bc[0], yd = b.y[i] - bc[1], zd = b.z[i] - bc[2];
        min_image(xd, yd, zd, W);
        x = float(xd);
        y = float(yd);
        z = float(zd);
        const bool fr = s.frozen[i] != 0;
        lim = float(fr ? rz2 : rl2) + margin;
        return fr;
    };
    auto within = [&](int j, float x, float y, float z, float lim, int f) {
        float dx = x - gx[f], dy = y - gy[f], dz = z - gz[f];
        dx -= L0 * rintf(dx * i0);
        dy -= L1 * rintf(dy * i1);
        dz -= L2 * rintf(dz * i2);
        return dx * dx + dy * dy + dz * dz <= lim && L.fid[f] != j;
    };
    int nz = 0, nfree = 0;
    for (int c0 = 0; c0 < nc; c0 += kBlock) {
        const int c = c0 + tid;
        const bool has = c < nc;
        const int j = has ? cand[c] : 0;
        float x, y, z, lim;
        const bool fr = place(j, x, y, z, lim);
        unsigned long long m[kFzLanes] = {};
        const int word = (c0 >> 6) + wave;
        for (int f0 = 0; f0 < nf; f0 += kFzLanes) {
#pragma unroll
            for (int q = 0; q < kFzLanes; ++q) {
                const int f = f0 + q < nf ? f0 + q : 0;
                const bool hit = has && f0 + q < nf && within(j, x, y, z, lim, f);
                const unsigned long long bal = __ballot(hit);
                if (lane == 0 && word < ncw && f0 + q < strip) bits[f * ncw + word] = bal;
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
            b.zmark[W.off + j] = 1;
        }
        nz += tot;
        nfree += totf;
        __syncthreads();  // the next round reuses the scratch rows
    }
    if (nz > kSlots) return false;
    // the free atoms' lists from their hit words, one (atom, word) per thread
    for (int s0 = 0; s0 < nf; s0 += strip) {
        const int ns = min(strip, nf - s0);
        if (s0 > 0) {  // the words of the next strip; its members' slots are in cand
            __syncthreads();
            for (int c0 = 0; c0 < nc; c0 += kBlock) {
                const int c = c0 + tid, word = (c0 >> 6) + wave;
                const bool has = c < nc && cand[c] != 0xFFFF;
                const int j = has ? R.slot[(size_t)w * kSlots + cand[c]] : 0;
                float x, y, z, lim;
                (void)place(j, x, y, z, lim);
                for (int f = 0; f < ns; ++f) {
                    const unsigned long long bal = __ballot(has && within(j, x, y, z, lim, s0 + f));
                    if (lane == 0 && word < ncw) bits[f * ncw + word] = bal;
                }
            }
            __syncthreads();
        }
        for (int t = tid; t < ns * ncw; t += kBlock) {
            const int k = t / ncw, wd = t - k * ncw, f = s0 + k;
            const unsigned long long *bw = bits + k * ncw;
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
    }
    // the order frozen slots are served in: classes of the number of free
    // atoms in reach, ascending slots within a class, so that the lanes of a
    // wavefront loop about equally long
    {
        unsigned long long *mask = R.mask + (size_t)w * kSlots * kFzLanes;
        constexpr int kRounds = kSlots / kBlock;
        int *cnt = reinterpret_cast<int *>(L.pool);  // [kRounds][kWaves][kClass], the candidates are done
        int cls[kRounds], rank[kRounds];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const int k = r * kBlock + tid;
            int c = -1;
            if (k < nz) {
                int pc = 0;
                for (int q = 0; q < kFzLanes; ++q) pc += __popcll(mask[(size_t)k * kFzLanes + q]);
                c = pc == 0 ? -1 : min(kClass - 1, pc / 6);  // no bits: a free slot
            }
            cls[r] = c;
            for (int v = 0; v < kClass; ++v) {
                const unsigned long long bal = __ballot(c == v);
                if (lane == 0) cnt[(r * kWaves + wave) * kClass + v] = __popcll(bal);
                if (c == v) rank[r] = __popcll(bal & ((1ull << lane) - 1ull));
            }
        }
        __syncthreads();
        for (int r = 0; r < kRounds; ++r) {
            if (cls[r] < 0) continue;
            int at = rank[r];
            for (int g = 0; g < kRounds * kWaves; ++g)
                for (int v = 0; v < kClass; ++v)
                    if (v < cls[r] || (v == cls[r] && g < r * kWaves + wave)) at += cnt[g * kClass + v];
            R.task[(size_t)w * kSlots + at] = uint16_t(r * kBlock + tid);
        }
    }
    for (int f = tid; f < nf; f += kBlock) {
        R.ref[((size_t)w * 3 + 0) * kFree + f] = L.fx[f];
        R.ref[((size_t)w * 3 + 1) * kFree + f] = L.fy[f];
        R.ref[((size_t)w * 3 + 2) * kFree + f] = L.fz[f];
    }
    if (tid == 0) {
        R.n[w] = nz;
        b.nz[w] = nz;
        atomicAdd(b.rebuild_count, 1ull);
    }
    __syncthreads();
    return true;
}

// starts of the free atoms' lists from their lengths (one wavefront)
template <int KIND>
__device__ inline void res_offsets(const int *fcnt, int nf)
{
    ResLds<KIND> &L = res_lds<KIND>();
    if (threadIdx.x >= 64) return;
    const int lane = threadIdx.x;
    int before = 0;
    for (int f0 = 0; f0 < nf; f0 += 64) {
        const int v = f0 + lane < nf ? fcnt[f0 + lane] : 0;
        int x = v;
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(x, o);
            if (lane >= o) x += t;
        }
        if (f0 + lane < nf) L.fofs[f0 + lane] = before + x - v;
        before += __shfl(x, 63);
    }
    if (lane == 0) L.fofs[nf] = before;
}

// energies of the atoms outside the zone (fixed parts only: no free atom is
// in their reach), in index order per thread
template <int KIND>
__device__ __attribute__((noinline)) void res_outside(const ResArgs *args, int nz, int prec)
{
    ResLds<KIND> &L = res_lds<KIND>();
    const BatchDev b = load_uniform(&args->b);
    const WalkerDev W = load_uniform(b.walkers + blockIdx.x);
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
    }
    __syncthreads();
}

// one evaluation at the free positions in LDS: forces of the free atoms and
// the walker's energy record
template <typename T, int KIND>
__device__ __attribute__((noinline)) void res_eval(const ResArgs *args, int nf, int nz)
{
    ResLds<KIND> &L = res_lds<KIND>();
    const BatchDev b = load_uniform(&args->b);
    const WalkerDev W = load_uniform(b.walkers + blockIdx.x);
    constexpr int prec = sizeof(T) == 8 ? 1 : 0;
    constexpr int kIlp = sizeof(T) == 8 ? kFreeIlp64 : kFreeIlp;
    const int w = blockIdx.x, tid = threadIdx.x;
    const SCCoef<T> c1 = sc_coef<T>(load_uniform(&b.field->sc[0]));
    const double rc2 = load_uniform(&b.field->rc2);
    const int ns = load_uniform(&b.field->nspec);
    const ResidentDev &R = b.r;
    const int S = slot_stride(nz);
    const double *rx = L.pool, *ry = rx + S, *rz = ry + S;
    double *rd = L.pool + 3 * S;       // density per slot, then 1/sqrt(rho)
    T *rw = reinterpret_cast<T *>(rd);  // in the low half for FP32
    constexpr int kRw = 8 / sizeof(T);
    double many = 0.0, pair = 0.0;
    // frozen slots: four lanes each, one mask word per lane, kFzIlp of its
    // free atoms at a time; the next slot's loads go out before this one's
    const unsigned long long *mask = R.mask + (size_t)w * kSlots * kFzLanes;
    const uint16_t *task = R.task + (size_t)w * kSlots, *slot = R.slot + (size_t)w * kSlots;
    {
        constexpr int kPer = kBlock / kFzLanes;
        const int nt = nz - nf, q = tid % kFzLanes;
        int t = tid / kFzLanes;
        int sn = t < nt ? task[t] : 0, s2 = t + kPer < nt ? task[t + kPer] : 0;
        unsigned long long mn = mask[sn * kFzLanes + q];
        int in = W.off + slot[sn];
        for (; t < nt; t += kPer) {
            unsigned long long m = mn;
            const int i = in, sl = sn;
            const double brho = R.base_rho[prec][i], bep = R.base_ep[prec][i];
            sn = s2;
            mn = mask[sn * kFzLanes + q];
            in = W.off + slot[sn];
            s2 = t + 2 * kPer < nt ? task[t + 2 * kPer] : 0;
            const double xi = rx[sl], yi = ry[sl], zi = rz[sl];
            double rho = 0.0, ep = 0.0;
            while (m) {
                double px[kFzIlp], py[kFzIlp], pz[kFzIlp];
                bool ok[kFzIlp];
                const SCPairDev *p[kFzIlp];
#pragma unroll
                for (int u = 0; u < kFzIlp; ++u) {
                    ok[u] = m != 0ull;
                    const int f = ok[u] ? kFzLanes * (__ffsll((long long)m) - 1) + q : 0;
                    m &= m - 1ull;
                    px[u] = L.fx[f];
                    py[u] = L.fy[f];
                    pz[u] = L.fz[f];
                    p[u] = KIND == 1 ? nullptr : L.tab + L.zt[sl] * ns + L.zt[L.fslot[f]];
                }
                add_density<T, KIND, kFzIlp>(W, rc2, c1, p, xi, yi, zi, px, py, pz, ok, rho, ep);
            }
            rho = row_sum<kFzLanes>(rho) + brho;
            ep = row_sum<kFzLanes>(ep) + bep;
            if (q == 0) {
                rd[sl] = rho;
                pair += ep;
            }
        }
    }
    // free atoms: kFreeLanes lanes per list, entries strided over the lanes
    const int g = tid / kFreeLanes, sub = tid % kFreeLanes;
    constexpr int kGroups = kBlock / kFreeLanes, kBatch = kFreeLanes * kIlp;
    const uint16_t *glist = R.flist + (size_t)w * kFree * R.fcap;
    const uint16_t *llist = reinterpret_cast<const uint16_t *>(L.pool + 4 * S);
    const bool lists = lists_fit(L.fofs[nf], S);
    // the slots of entries k, k + kFreeLanes, ... of free atom f (-1: none)
    auto fetch = [&](int f, int k, int cnt, int (&e)[kIlp]) {
#pragma unroll
        for (int u = 0; u < kIlp; ++u) {
            const int kk = k + u * kFreeLanes;
            e[u] = -1;
            if (kk < cnt) e[u] = lists ? int(llist[L.fofs[f] + kk]) : int(glist[(size_t)f * R.fcap + kk]);
        }
    };
    for (int f = g; f < nf; f += kGroups) {
        const int cnt = L.fofs[f + 1] - L.fofs[f];
        const int sl = L.fslot[f], zt = L.zt[sl];
        const double xi = L.fx[f], yi = L.fy[f], zi = L.fz[f];
        double rho = 0.0, ep = 0.0;
        for (int k = sub; k < cnt; k += kBatch) {
            int e[kIlp];
            fetch(f, k, cnt, e);
            double px[kIlp], py[kIlp], pz[kIlp];
            bool ok[kIlp];
            const SCPairDev *p[kIlp];
#pragma unroll
            for (int u = 0; u < kIlp; ++u) {
                ok[u] = e[u] >= 0;
                const int j = ok[u] ? e[u] : sl;
                px[u] = rx[j];
                py[u] = ry[j];
                pz[u] = rz[j];
                p[u] = KIND == 1 ? nullptr : L.tab + zt * ns + L.zt[j];
            }
            add_density<T, KIND, kIlp>(W, rc2, c1, p, xi, yi, zi, px, py, pz, ok, rho, ep);
        }
        rho = row_sum<kFreeLanes>(rho);
        ep = row_sum<kFreeLanes>(ep);
        if (sub == 0) {
            rd[sl] = rho;
            pair += ep;
        }
    }
    __syncthreads();
    // embedding energies and 1/sqrt(rho), a slot per thread
    for (int k = tid; k < nz; k += kBlock) {
        const double rho = rd[k], r = sqrt(rho);
        many -= r;
        rw[kRw * k] = rho < 1.0e-8 ? T(-1) : T(1.0 / r);
    }
    __syncthreads();
    // forces of the free atoms (the expressions of the chain's pass 2)
    for (int f = g; f < nf; f += kGroups) {
        const int cnt = L.fofs[f + 1] - L.fofs[f];
        const int sl = L.fslot[f], zt = L.zt[sl];
        const double xi = L.fx[f], yi = L.fy[f], zi = L.fz[f];
        const T isi = rw[kRw * sl];
        double fx = 0.0, fy = 0.0, fz = 0.0;
        for (int k = sub; k < cnt; k += kBatch) {
            int e[kIlp];
            fetch(f, k, cnt, e);
            double dx[kIlp], dy[kIlp], dz[kIlp], r2[kIlp];
            T isj[kIlp];
            bool in[kIlp];
            const SCPairDev *p[kIlp];
#pragma unroll
            for (int u = 0; u < kIlp; ++u) {
                const int j = e[u] >= 0 ? e[u] : sl;
                dx[u] = xi - rx[j];
                dy[u] = yi - ry[j];
                dz[u] = zi - rz[j];
                isj[u] = rw[kRw * j];
                p[u] = KIND == 1 ? nullptr : L.tab + zt * ns + L.zt[j];
                min_image(dx[u], dy[u], dz[u], W);
                r2[u] = dx[u] * dx[u] + dy[u] * dy[u] + dz[u] * dz[u];
                in[u] = e[u] >= 0 && r2[u] <= rc2 && r2[u] > 1.0e-16;
            }
            T ir2[kIlp], un[kIlp], um[kIlp];
            pair_terms<T, KIND, kIlp>(r2, in, c1, p, ir2, un, um);
#pragma unroll
            for (int u = 0; u < kIlp; ++u) {
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
        fx = row_sum<kFreeLanes>(fx);
        fy = row_sum<kFreeLanes>(fy);
        fz = row_sum<kFreeLanes>(fz);
        if (sub == 0) {
            const int i = W.off + L.fid[f];
            b.fx[i] = fx;
            b.fy[i] = fy;
            b.fz[i] = fz;
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

// the walker's state machine
template <int KIND>
__device__ __attribute__((noinline)) void res_step(const ResArgs *args, int nf)
{
    ResLds<KIND> &L = res_lds<KIND>();
    const BatchDev b = load_uniform(&args->b);
    const SearchDev s = load_uniform(&args->s);
    const WalkerDev *W = b.walkers + blockIdx.x;
    Ctx C_{b, s, load_uniform(&W->off), load_uniform(&W->n), b.A, nf, L.pool};
    // the walker's scalars are private to each thread during its step (all
    // threads take the same branches) and in LDS during the evaluations
    WalkerState w = L.ws;
    walker_step(C_, w, L.sh);
    __syncthreads();
    if (threadIdx.x == 0) L.ws = w;
}

// the walker goes over to the chain: a fresh zone, full evaluations first
__device__ inline void leave(const BatchDev &b, const SearchDev &s, int w)
{
    b.zflag[w] = AKMC_ZONE_FRESH;
    b.rebuild[w] = 1;
    s.ws[w].res |= AKMC_RES_LEFT;
}

// Micro-steps of resident walkers, one workgroup each.  service: the chain
// has just run, and with it k_res_base for the walkers on their first
// micro-step; from then on a walker needs nothing from outside.  nsteps 0:
// only the first list build of the walkers just started, at the probes of
// their first micro-step, so that a walker that does not fit is on the chain
// before that step.  (Not a kernel of its own: LDS that out-of-line functions
// share between kernels is no longer addressed directly.)
template <int KIND>
__global__ void __launch_bounds__(kBlock, 4) k_search_resident(const ResArgs *args, int nsteps, int logic, int service)
{
    ResLds<KIND> &L = res_lds<KIND>();
    const BatchDev b = load_uniform(&args->b);
    const SearchDev s = load_uniform(&args->s);
    const int wid = blockIdx.x, tid = threadIdx.x;
    int flags = b.zflag[wid];
    if (!(flags & AKMC_ZONE_RES) || b.active[wid] == 0) return;
    if (tid == 0) {
        L.ws = s.ws[wid];
        L.ws.res &= ~AKMC_RES_WAITS;
    }
    if constexpr (KIND != 1) stage_sc_table(*b.field, L.tab);
    __syncthreads();
    if (L.ws.kind == WK_IDLE || L.ws.state == ST_DONE) return;
    const WalkerDev W = load_uniform(b.walkers + wid);
    const int nf = s.nact[wid];
    if (nf < 1 || nf > kFree) return;  // (the host admits no such walker)
    const double h2 = b.field->half_skin2;
    int nz = b.r.n[wid], evals32 = 0, eok = b.r.eok[wid];
    if (nz >= 0) {
        for (int f = tid; f < nf; f += kBlock) L.fslot[f] = b.r.fslot[wid * kFree + f];
        res_offsets<KIND>(b.r.fcnt + wid * kFree, nf);
    }
    for (int f = tid; f < nf; f += kBlock) L.fid[f] = uint16_t(s.act[W.off + f] - W.off);
    if (nsteps == 0) {
        if (nz >= 0) return;
        for (int f = tid; f < nf; f += kBlock) {
            const int i = s.act[W.off + f];
            L.fx[f] = b.x[i];
            L.fy[f] = b.y[i];
            L.fz[f] = b.z[i];
        }
        __syncthreads();
        if (!res_build<KIND>(args, nf) && tid == 0) leave(b, s, wid);
        return;
    }
    bool loaded = false, too_big = false;  // loaded: the zone's records are in the pool
    for (int step = 0; step < nsteps; ++step) {
        __syncthreads();
        if (L.ws.state == ST_DONE) break;
        // the mode the state machine left the walker in (BatchDev.active)
        const int mode = step == 0 ? b.active[wid]
                                   : (L.ws.kind == WK_VERIFY || L.ws.state == ST_R_E64) ? 2 : s.default_mode;
        const int prec = mode == 2 ? 1 : 0;
        const int full = prec ? AKMC_ZONE_FULL64 : AKMC_ZONE_FULL32;
        if (step == 0 && service) {  // the fixed parts that k_res_base has just made
            const int made = flags & (akmc_res_precisions(s) | full);
            flags &= ~made;
            if (made & AKMC_ZONE_FULL32) eok &= ~1;
            if (made & AKMC_ZONE_FULL64) eok &= ~2;
        }
        if (flags & full) {
            if (tid == 0) L.ws.res |= AKMC_RES_WAITS;
            break;
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
            if (!res_build<KIND>(args, nf)) {
                too_big = true;
                break;
            }
            nz = b.r.n[wid];
            res_offsets<KIND>(b.r.fcnt + wid * kFree, nf);
            __syncthreads();
            eok = 0;
            loaded = false;
        }
        if (!(eok & (1 << prec))) {
            res_outside<KIND>(args, nz, prec);
            eok |= 1 << prec;
            loaded = false;
        }
        const int S = slot_stride(nz);
        if (!loaded) {
            for (int k = tid; k < nz; k += kBlock) {
                const int i = W.off + b.r.slot[(size_t)wid * kSlots + k];
                L.pool[k] = b.x[i];
                L.pool[S + k] = b.y[i];
                L.pool[2 * S + k] = b.z[i];
                L.zt[k] = uint8_t(b.type[i]);
            }
            if (lists_fit(L.fofs[nf], S)) {
                uint16_t *llist = reinterpret_cast<uint16_t *>(L.pool + 4 * S);
                const int lane = tid & 63;
                for (int f = tid >> 6; f < nf; f += kWaves) {
                    const uint16_t *gl = b.r.flist + ((size_t)wid * kFree + f) * b.r.fcap;
                    const int o = L.fofs[f], n = L.fofs[f + 1] - o;
                    for (int k = lane; k < n; k += 64) llist[o + k] = gl[k];
                }
            }
            loaded = true;
        } else {
            for (int f = tid; f < nf; f += kBlock) {
                const int k = L.fslot[f];
                L.pool[k] = L.fx[f];
                L.pool[S + k] = L.fy[f];
                L.pool[2 * S + k] = L.fz[f];
            }
        }
        __syncthreads();
        if (prec) res_eval<double, KIND>(args, nf, nz);
        else res_eval<float, KIND>(args, nf, nz);
        if (!logic) break;
        evals32 += mode == 1;
        if (L.ws.kind == WK_VERIFY) loaded = false;  // its Lanczos vectors take the pool
        res_step<KIND>(args, nf);
    }
    __syncthreads();
    if (tid == 0) {
        b.zflag[wid] = flags;
        b.r.eok[wid] = eok;
        if (logic) s.ws[wid] = L.ws;
        s.evals32[wid] += evals32;
        if (too_big) leave(b, s, wid);
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

// (one pass over the lists for both precisions: the list and position loads
// bound it)
template <int KIND, bool F32, bool F64>
__device__ inline void res_base_atoms(const BatchDev &b, const WalkerDev &W, const SCPairDev *tab)
{
    const FieldDev &F = *b.field;
    const SCCoef<float> c32 = sc_coef<float>(F.sc[0]);
    const SCCoef<double> c64 = sc_coef<double>(F.sc[0]);
    const int sub = threadIdx.x % kBaseLanes;
    constexpr int per = kBaseBlock / kBaseLanes;
    for (int l = blockIdx.y * per + (int)threadIdx.x / kBaseLanes; l < W.n; l += kBaseSplit * per) {
        const int i = W.off + l, cnt = b.nnb[i];
        const double xi = b.x[i], yi = b.y[i], zi = b.z[i];
        Sum2 sum[4] = {};  // density, half pair energy; FP32, FP64
        for (int k = sub; k < cnt; k += kBaseLanes) {
            const int j = W.off + int(nbr_entry(b, k, i) & AKMC_NB_JMASK);
            const bool ok[1] = {b.zfrozen[j] != 0};
            const double px[1] = {b.x[j]}, py[1] = {b.y[j]}, pz[1] = {b.z[j]};
            const SCPairDev *p[1] = {KIND == 1 ? nullptr : tab + b.type[i] * F.nspec + b.type[j]};
            if constexpr (F32) {
                double r = 0.0, e = 0.0;
                add_density<float, KIND, 1>(W, F.rc2, c32, p, xi, yi, zi, px, py, pz, ok, r, e);
                sum[0].add(r);
                sum[1].add(e);
            }
            if constexpr (F64) {
                double r = 0.0, e = 0.0;
                add_density<double, KIND, 1>(W, F.rc2, c64, p, xi, yi, zi, px, py, pz, ok, r, e);
                sum[2].add(r);
                sum[3].add(e);
            }
        }
#pragma unroll
        for (int v = F32 ? 0 : 2; v < (F64 ? 4 : 2); ++v)
            for (int o = kBaseLanes / 2; o > 0; o >>= 1) {
                const double h = __shfl_xor(sum[v].h, o), lo = __shfl_xor(sum[v].l, o);
                sum[v].add(h);
                sum[v].l += lo;
            }
        if (sub == 0) {
            if constexpr (F32) {
                b.r.base_rho[0][i] = sum[0].h + sum[0].l;
                b.r.base_ep[0][i] = sum[1].h + sum[1].l;
            }
            if constexpr (F64) {
                b.r.base_rho[1][i] = sum[2].h + sum[2].l;
                b.r.base_ep[1][i] = sum[3].h + sum[3].l;
            }
        }
    }
}

// The parts of every atom's density and pair energy that come from frozen
// neighbours, for the resident walkers on their first micro-step (kBaseSplit
// workgroups per walker), in every precision that the searches may come to: a
// search goes over to FP64 at its verification, and with these parts at hand
// it does so without waiting for an evaluation of the chain.  (When
// verification is turned on under running searches the FP64 parts follow with
// the next chunk, from the same lists: frozen atoms do not move.)
template <int KIND>
__global__ void __launch_bounds__(kBaseBlock) k_res_base(BatchDev b, int precisions)
{
    __shared__ SCPairDev tab[KIND == 1 ? 1 : kResSpec * kResSpec];
    const int w = blockIdx.x, mode = b.active[w], f = b.zflag[w];
    const int todo = f & (precisions | (mode == 2 ? AKMC_ZONE_FULL64 : AKMC_ZONE_FULL32)) &
                     (AKMC_ZONE_FULL32 | AKMC_ZONE_FULL64);
    if (mode == 0 || !(f & AKMC_ZONE_RES) || !todo) return;
    if constexpr (KIND != 1) stage_sc_table(*b.field, tab);
    const WalkerDev W = b.walkers[w];
    if (!(todo & AKMC_ZONE_FULL64)) res_base_atoms<KIND, true, false>(b, W, tab);
    else if (!(todo & AKMC_ZONE_FULL32)) res_base_atoms<KIND, false, true>(b, W, tab);
    else res_base_atoms<KIND, true, true>(b, W, tab);
}

}  // namespace

void akmc_launch_res_base(const BatchDev &b, const FieldDev &hf, int precisions, hipStream_t st)
{
    const dim3 g(b.W, kBaseSplit);
    switch (akmc_sc_kind(hf)) {
    case 1: k_res_base<1><<<g, kBaseBlock, 0, st>>>(b, precisions); break;
    case 2: k_res_base<2><<<g, kBaseBlock, 0, st>>>(b, precisions); break;
    default: k_res_base<0><<<g, kBaseBlock, 0, st>>>(b, precisions);
    }
}

void akmc_launch_search_resident(int nwalkers, const FieldDev &hf, const ResArgs *args, int nsteps, int logic,
                                 int service, hipStream_t st)
{
    switch (akmc_sc_kind(hf)) {
    case 1: k_search_resident<1><<<nwalkers, kBlock, 0, st>>>(args, nsteps, logic, service); break;
    case 2: k_search_resident<2><<<nwalkers, kBlock, 0, st>>>(args, nsteps, logic, service); break;
    default: k_search_resident<0><<<nwalkers, kBlock, 0, st>>>(args, nsteps, logic, service);
    }
}

void akmc_launch_res_admit(int nwalkers, const FieldDev &hf, const ResArgs *args, hipStream_t st)
{
    akmc_launch_search_resident(nwalkers, hf, args, 0, 0, 0, st);
}
