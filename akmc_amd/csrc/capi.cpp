// C ABI of libakmc_hip.so: potentials text, field setup and walker batches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cctype>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <memory>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/akmc.h"
#include "akmc_internal.h"

namespace {

// e^2/(4 pi eps0) in eV A, the value with which the reference reproduces
// its own example energy (docs/examples/gdc/basis:3)
constexpr double kCTOEV = 14.3997584;
constexpr double kPI = 3.14159265358979323846;

thread_local std::string g_err;

int fail(int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

#define HIPCHK(expr)                                                                          \
    do {                                                                                      \
        hipError_t e_ = (expr);                                                               \
        if (e_ != hipSuccess) return fail(AKMC_EHIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

std::vector<std::string> split_ws(const std::string &s)
{
    std::istringstream is(s);
    std::vector<std::string> w;
    std::string t;
    while (is >> t) w.push_back(t);
    return w;
}

std::string lower(std::string s)
{
    for (auto &c : s) c = (char)std::tolower((unsigned char)c);
    return s;
}

struct SpeciesRec {
    std::string name;
    double mass, charge;
};
struct SCPot {
    std::string A, B;
    double eps, a, n, m, c;
};
// a two-body entry: form (IonForm) and its parameters in the order of the
// potentials text (TwoBody.cpp:98-245)
struct BuckPot {
    std::string A, B;
    double Ab, rho, C;
    int form = 0;
    double par[6] = {0, 0, 0, 0, 0, 0};
};
// a tabulated EAM potential as readLEAM leaves it
// (potentials/metal/MetalPotential.cpp:276-361)
struct EamPot {
    std::string A, B, file;
    int nrho = 0, nr = 0;
    double drho = 0, dr = 0, cut = 0;
    std::vector<double> F, rho, phi;  // embedding, density, pair (the file's r phi divided by r)
};

}  // namespace

struct akmc_field_s {
    int kind = -1;  // 0 many-body, 1 ionic
    double rc = 0.0;
    bool min_image = true;
    bool nbrlist = false;
    double verlet_shell = 1.0;
    int do_ewald = 1;  // pair default (potentials/pair/Field.h:28)
    double madelung_acc = 1.0e-6;
    bool explicit_ewald = false;
    double eta = 0.0;
    int gcell[3] = {0, 0, 0};
    double skin = 0.7;  // best of a 0.45-1.6 A sweep on the batched dimer workload
    double list_density = 0.0;  // atoms per A^3 the neighbour lists are sized for (0: each walker's N / V)
    std::vector<SpeciesRec> species;
    std::vector<SCPot> sc;
    std::vector<BuckPot> buck;
    std::vector<EamPot> eam;
    double2 *eam_dev = nullptr;  // device copy of every EAM table (one allocation)
    double dsf_alpha = 0.0;      // ewald damp: the damping of the shifted Coulomb sum
    double *dsf_dev = nullptr;   // its erfc mesh on the device (energy, force terms)
    FieldDev host{};
    FieldDev *dev = nullptr;
    int table[AKMC_MAXPAIR];
    // cached single-walker batch behind akmc_field_forces
    akmc_batch_t single = nullptr;
    int single_n = -1;
    double single_lat[9] = {0};
    int nk_last = 0;
    int fp64 = 0;
};

struct akmc_batch_s {
    akmc_field_t f = nullptr;
    int W = 0, A = 0;
    std::vector<WalkerDev> hw;
    std::vector<int> hk_n;       // [3][nk]
    std::vector<double> hk_v, hg0, hg1;
    BatchDev d{};
    hipStream_t stream = nullptr;
    std::vector<void *> allocs;
    std::vector<WalkerOut> hout;
    // what a force call sends and gets back lies together on the device: x, y,
    // z, type, rebuild and active flags, q; then forces, energy records and
    // the overflow flag.  Small batches move each part in one transfer through
    // pinned memory.
    char *io = nullptr, *io_pin = nullptr;
    size_t io_pin_n = 0;
    size_t io_q = 0, io_in = 0, io_out = 0, io_end = 0;
    // LDS staging of the many-body pair kernels is possible when every
    // walker's gather records fit one workgroup's LDS
    bool stage_ok = false;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    unsigned long long rebuild_base = 0;
    // search state
    SearchDev s{};
    bool search_alloc = false;
    std::vector<WalkerState> hws;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    int graph_steps = 0;
    SearchDev graph_args{};  // kernel arguments baked into the captured graph
    BatchDev graph_d{};
    int graph_prec = 0;
    bool use_graphs = true;
    // HIP events around the FP32 Sutton-Chen pass-2 launch of every
    // micro-step of akmc_batch_run (kernel timer)
    static constexpr int kTimerSteps = 64;
    bool ktimer = false;
    hipEvent_t kev[2][kTimerSteps] = {};
    double kms = 0.0;
    long long klaunches = 0;
    double *basin = nullptr;  // [3][A] saved search positions
    hipEvent_t evp[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    // host copy of the frozen mask and the per-walker free-atom lists
    std::vector<int> hfrozen, hact, hnact;
    // active zones of the search micro-steps (BatchDev.zflag ...): on by
    // default for minimum-image Sutton-Chen fields
    bool zone_on = true;
    // the batch's largest walker has at least kWideLogicAtoms atoms
    bool logic_wide = false;
    int *zflag = nullptr, *zmark = nullptr, *zlist = nullptr, *nz = nullptr;
    std::vector<int> hzflag;
    // resident searches (search_resident.hip): their buffers (res_none: no
    // memory for them, so every walker takes the chain)
    ResidentDev r{};
    bool res_none = false;
    bool res_on = true;               // akmc_batch_set_resident
    int *zf_pin = nullptr;            // zflag after the last starts (pinned)
    ResArgs *res_args = nullptr;      // device copy of the descriptors its kernel
    ResArgs res_host{};               // reads, and what it holds
    int graph_res = 0;
    // kernel variants of the search micro-steps' Sutton-Chen passes:
    // (lanes, unroll, staged) of pass 1, of pass 2, then of the FP64 passes
    // of mixed steps; lanes 0: the default
    int sv[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    // work lists of the search micro-steps' pair kernels and their grids
    int2 *wl_tab[4] = {nullptr, nullptr, nullptr, nullptr};
    int *wl_count = nullptr;
    int wl_grid_staged = 0, wl_grid_plain = 0;
    // pinned status staging: one stream sync per host check of a run
    WalkerState *hws_pin = nullptr;
    int *ov_pin = nullptr;
    char *gat_pin = nullptr;    // pinned / device index lists and packed output
    char *gat_dev = nullptr;    // of akmc_batch_get_walkers_* (gather kernel)
    size_t gat_n = 0;
    int inflight = 0;           // a chunk launched by akmc_batch_run_async awaits its wait
    int inflight_steps = 0;
    char *desc_dev = nullptr;   // device buffer of akmc_batch_descriptors (grows to the largest call)
    size_t desc_n = 0;
    void *stage_pin = nullptr;  // pinned host / device staging of walker starts
    void *stage_dev = nullptr;
    size_t stage_n = 0;
    // the fresh states of started walkers (one pinned transfer per start);
    // each pinned buffer is rewritten only after its last transfer is done
    StartItem *st_pin = nullptr, *st_dev = nullptr;
    hipEvent_t stage_ev = nullptr, st_ev = nullptr;
    bool stage_pending = false, st_pending = false;
    // starts queued behind a chunk in flight: their states replace that
    // chunk's status copy when it is waited for
    std::vector<std::pair<int, WalkerState>> started_inflight;
    // reads of ended walkers while a chunk is in flight
    hipStream_t side = nullptr;
    // harvest: each chunk ends by copying the positions of the walkers that
    // ended in it into one of two mapped host buffers ([3][A] each), in turn
    int hv_on = 0, hv_cur = 0, hv_inflight = -1, hv_last = -1;
    int *harvested = nullptr;
    double *hv_pin[2] = {nullptr, nullptr}, *hv_dev[2] = {nullptr, nullptr};
};

namespace {

// readParameters (MetalPotential.cpp:363-386): whole lines of numbers until
// n values are in; numbers past n on the last line are dropped (the
// reference writes them past its array)
bool read_values(std::istream &in, int n, std::vector<double> &out)
{
    out.clear();
    std::string line;
    while ((int)out.size() < n) {
        if (!std::getline(in, line)) return false;
        for (const std::string &w : split_ws(line)) {
            if ((int)out.size() >= n) break;
            out.push_back(std::stod(w));
        }
    }
    return true;
}

// readLEAM (MetalPotential.cpp:276-361): four comment/element lines,
// "Nrho drho Nr dr cutoff", one element line, then F(rho) on the rho mesh,
// rho(r) and r phi(r) on the r mesh; phi_i = (r phi)_i / (i dr), so the
// first entry is the file's value / 0 as in the reference.
int read_lammps_eam(EamPot &p)
{
    std::ifstream in(p.file);
    if (!in) return fail(AKMC_EINVAL, "could not find LAMMPS style EAM file %s", p.file.c_str());
    std::string line;
    try {
        for (int k = 0; k < 4; ++k)
            if (!std::getline(in, line)) throw std::runtime_error("header");
        if (!std::getline(in, line)) throw std::runtime_error("mesh line");
        auto w = split_ws(line);
        p.nrho = std::stoi(w.at(0));
        p.drho = std::stod(w.at(1));
        p.nr = std::stoi(w.at(2));
        p.dr = std::stod(w.at(3));
        p.cut = std::stod(w.at(4));
        if (p.nrho < 2 || p.nr < 2 || !(p.drho > 0) || !(p.dr > 0))
            return fail(AKMC_EINVAL, "EAM file %s: bad mesh line", p.file.c_str());
        if (!std::getline(in, line)) throw std::runtime_error("element line");
        if (!read_values(in, p.nrho, p.F) || !read_values(in, p.nr, p.rho) || !read_values(in, p.nr, p.phi))
            throw std::runtime_error("tables");
    } catch (const std::exception &) {
        return fail(AKMC_EINVAL, "EAM file %s is truncated or malformed", p.file.c_str());
    }
    for (int i = 0; i < p.nr; ++i) p.phi[i] = p.phi[i] / (i * p.dr);
    return AKMC_SUCCESS;
}

int parse_potentials(akmc_field_t f, const char *text)
{
    std::istringstream in(text ? text : "");
    std::string line;
    bool closed = false;
    auto next_line = [&](std::string &l) -> bool {
        while (std::getline(in, l)) {
            if (!split_ws(l).empty()) return true;
        }
        return false;
    };
    while (next_line(line)) {
        auto w = split_ws(lower(line));
        const std::string &k = w[0];
        try {
            if (k == "cutoff") {
                f->rc = std::stod(w.at(1));
            } else if (k == "nbrlist") {
                f->nbrlist = true;
                f->verlet_shell = std::stod(w.at(1));
            } else if (k == "noimage") {
                f->min_image = false;
            } else if (k == "ewald") {
                const std::string &sub = w.at(1);
                if (sub == "precis") {
                    f->do_ewald = 1;
                    f->madelung_acc = std::stod(w.at(2));
                } else if (sub == "damp") {
                    // damped-shifted Coulomb with damping alpha (pair Field.cpp:265-270)
                    f->do_ewald = 2;
                    f->dsf_alpha = std::stod(w.at(2));
                } else if (sub == "none") {
                    f->do_ewald = 0;
                } else {
                    return fail(AKMC_EUNSUPPORTED, "ewald %s is not supported on the device", sub.c_str());
                }
            } else if (k == "species") {
                int n = std::stoi(w.at(1));
                for (int s = 0; s < n; ++s) {
                    std::string sl;
                    if (!next_line(sl)) return fail(AKMC_EINVAL, "species: missing line");
                    auto sw = split_ws(sl);  // species lines keep their case (Species.cpp:45-60)
                    f->species.push_back({sw.at(0), std::stod(sw.at(1)), std::stod(sw.at(2))});
                }
            } else if (k == "many" || k == "manybody") {
                f->kind = 0;
                int n = std::stoi(w.at(1));
                for (int p = 0; p < n; ++p) {
                    std::string kl, pl;
                    if (!next_line(kl) || !next_line(pl)) return fail(AKMC_EINVAL, "manybody: missing lines");
                    std::string key = lower(split_ws(kl).at(0));
                    auto pw = split_ws(pl);
                    if (key == "eam") {
                        // A B file [lammps|dlpoly] (ManyBody.cpp:269-307)
                        EamPot e;
                        e.A = pw.at(0);
                        e.B = pw.at(1);
                        e.file = pw.at(2);
                        std::string fmt = pw.size() > 3 ? pw[3] : "lammps";
                        if (fmt == "dlpoly")
                            return fail(AKMC_EUNSUPPORTED, "the DL_POLY tabulated EAM format is not supported");
                        if (fmt != "lammps") return fail(AKMC_EINVAL, "unrecognised EAM format");
                        const int rc = read_lammps_eam(e);
                        if (rc != AKMC_SUCCESS) return rc;
                        f->eam.push_back(std::move(e));
                    } else if (key == "suttonchen") {
                        // A B eps a n m c (ManyBody.cpp:148-163)
                        f->sc.push_back({pw.at(0), pw.at(1), std::stod(pw.at(2)), std::stod(pw.at(3)),
                                         std::stod(pw.at(4)), std::stod(pw.at(5)), std::stod(pw.at(6))});
                    } else {
                        return fail(AKMC_EUNSUPPORTED, "many-body form '%s' is not supported on the device",
                                    key.c_str());
                    }
                    if (!f->eam.empty() && !f->sc.empty())
                        return fail(AKMC_EINVAL, "many-body potential types can not be mixed");
                }
            } else if (k == "twobody") {
                f->kind = 1;
                int n = std::stoi(w.at(1));
                for (int p = 0; p < n; ++p) {
                    std::string kl, pl;
                    if (!next_line(kl) || !next_line(pl)) return fail(AKMC_EINVAL, "twobody: missing lines");
                    std::string key = lower(split_ws(kl).at(0));
                    // potenKey (TwoBody.cpp:440-470) and the parameter counts of loadPotential
                    int form = -1, npar = 0;
                    if (key == "buck") form = ION_BUCK, npar = 3;
                    else if (key == "morse") form = ION_MORSE, npar = 4;
                    else if (key == "ljones") form = ION_LJONES, npar = 2;
                    else if (key == "bhm") form = ION_BHM, npar = 5;
                    else if (key == "severnsix") form = ION_SEVNSIX, npar = 2;
                    if (form < 0)
                        return fail(AKMC_EUNSUPPORTED, "two-body form '%s' is not supported on the device",
                                    key.c_str());
                    auto pw = split_ws(pl);
                    BuckPot bp{pw.at(0), pw.at(1), 0.0, 1.0, 0.0};
                    bp.form = form;
                    for (int q = 0; q < npar; ++q) bp.par[q] = std::stod(pw.at(2 + q));
                    if (form == ION_BUCK) {  // A B A rho C (TwoBody.cpp:98-112)
                        bp.Ab = bp.par[0];
                        bp.rho = bp.par[1];
                        bp.C = bp.par[2];
                    }
                    f->buck.push_back(bp);
                }
            } else if (k == "close") {
                closed = true;
                break;
            } else if (k == "maxnbrs") {
                // accepted and ignored, as the reference can never match it
            } else {
                return fail(AKMC_EINVAL, "unrecognised key word used in potentials file %s", k.c_str());
            }
        } catch (const std::exception &) {
            return fail(AKMC_EINVAL, "malformed potentials line: %s", line.c_str());
        }
    }
    (void)closed;
    if (f->kind < 0) return fail(AKMC_EINVAL, "potentials text has no manybody or twobody section");
    if (f->species.empty()) return fail(AKMC_EINVAL, "potentials text has no species");
    if ((int)f->species.size() > AKMC_MAXSPEC) return fail(AKMC_ECAPACITY, "more than %d species", AKMC_MAXSPEC);
    if ((int)f->eam.size() > AKMC_MAXEAM) return fail(AKMC_ECAPACITY, "more than %d EAM tables", AKMC_MAXEAM);
    return AKMC_SUCCESS;
}

// species-pair tables: -1 default for many-body (ManyBody.cpp:869), 0 for
// pair potentials (TwoBody.cpp:509)
void build_tables(akmc_field_t f)
{
    int ns = (int)f->species.size();
    FieldDev &h = f->host;
    std::memset(&h, 0, sizeof h);
    h.kind = f->kind;
    h.nspec = ns;
    h.min_image = f->min_image ? 1 : 0;
    h.do_ewald = f->kind == 1 ? f->do_ewald : 0;
    h.rc = f->rc;
    h.rc2 = f->rc * f->rc;
    double rl = f->rc + f->skin;
    h.rlist2 = rl * rl;
    // between rebuilds an atom moves at most skin/2, so every atom that comes
    // within rc of a free atom was within rc + skin/2 of it at the rebuild
    const double rz = f->rc + 0.5 * f->skin + 1.0e-6;
    h.rzone2 = rz * rz;
    h.half_skin2 = 0.25 * f->skin * f->skin;
    // ionic lists put the first shells (r <= 3.5 A) first; the FP32 path
    // evaluates them in FP64
    h.rnear2 = f->kind == 1 ? (3.5 + f->skin) * (3.5 + f->skin) : 0.0;
    h.cfact = kCTOEV;
    for (int i = 0; i < AKMC_MAXPAIR; ++i) f->table[i] = f->kind == 0 ? -1 : 0;
    // EAM: species pair -> table, both orders (calculateEAMEnergyMesh,
    // ManyBody.cpp:937-1000); the device table pointers are set when the
    // tables are uploaded
    h.eam = f->eam.empty() ? 0 : 1;
    for (int i = 0; i < AKMC_MAXPAIR; ++i) h.eam_tab[i] = -1;
    for (int k = 0; k < (int)f->eam.size(); ++k)
        for (int i = 0; i < ns; ++i)
            for (int j = 0; j < ns; ++j)
                if (f->species[i].name == f->eam[k].A && f->species[j].name == f->eam[k].B) {
                    h.eam_tab[j * ns + i] = k;
                    h.eam_tab[i * ns + j] = k;
                }
    h.eam_one = 0;
    if (h.eam) {
        h.eam_one = 1;
        for (int i = 0; i < ns * ns; ++i) h.eam_one &= h.eam_tab[i] == h.eam_tab[0] && h.eam_tab[0] >= 0;
        for (int k = 0; k < (int)f->eam.size(); ++k) {
            const EamPot &e = f->eam[k];
            EamTabDev &t = h.eamt[k];
            t.nr = e.nr;
            t.nrho = e.nrho;
            t.dr = e.dr;
            t.drho = e.drho;
            t.cut = e.cut;
        }
    }
    for (int i = 0; i < ns; ++i)
        for (int j = 0; j < ns; ++j) {
            int np = f->kind == 0 ? (int)f->sc.size() : (int)f->buck.size();
            for (int k = 0; k < np; ++k) {
                const std::string &A = f->kind == 0 ? f->sc[k].A : f->buck[k].A;
                const std::string &B = f->kind == 0 ? f->sc[k].B : f->buck[k].B;
                if (f->species[i].name == A && f->species[j].name == B) {
                    f->table[j * ns + i] = k;
                    f->table[i * ns + j] = k;
                }
            }
        }
    for (int i = 0; i < ns; ++i)
        for (int j = 0; j < ns; ++j) {
            int k = f->table[i * ns + j];
            if (f->kind == 0) {
                SCPairDev &p = h.sc[i * ns + j];
                if (k < 0) continue;
                const SCPot &s = f->sc[k];
                p.on = 1;
                p.d = {s.a, s.n, s.m, s.eps, (s.eps * s.c) * (s.eps * s.c), s.n * s.eps,
                       0.5 * s.m * (s.eps * s.c) * (s.eps * s.c)};
                p.f = {(float)p.d.a, (float)p.d.n, (float)p.d.m, (float)p.d.eps, (float)p.d.rho_coef,
                       (float)p.d.fs_coef, (float)p.d.fm_coef};
                auto as_int = [](double e) { return (e >= 0 && e <= 64 && std::floor(e) == e) ? (int)e : -1; };
                p.n_int = as_int(s.n);
                p.m_int = as_int(s.m);
            } else {
                IonPairDev &p = h.ion[i * ns + j];
                if (k < 0 || k >= (int)f->buck.size()) continue;
                const BuckPot &b = f->buck[k];
                p.on = 1;
                p.form = b.form;
                p.Ad = b.Ab;
                p.inv_rhod = 1.0 / b.rho;
                p.Cd = b.C;
                p.A = (float)p.Ad;
                p.inv_rho = (float)p.inv_rhod;
                p.C = (float)p.Cd;
                for (int q = 0; q < 6; ++q) {
                    p.pd[q] = b.par[q];
                    p.pf[q] = (float)b.par[q];
                }
            }
        }
    h.all96 = f->kind == 0 && f->eam.empty() ? 1 : 0;
    for (int k = 0; k < ns * ns; ++k)
        h.all96 &= h.sc[k].on && h.sc[k].n_int == 9 && h.sc[k].m_int == 6 && h.sc[k].d.a > 0.0;
}

// lanes per atom and gathers in flight of the pair kernels for one cell of n
// atoms behind the plain force call.  Below two wavefronts per SIMD at 8
// lanes (16,384 atoms) a wavefront per atom: 255 atoms 65 + 56 us at one lane,
// 7 + 6 us so; above, 8 lanes: 31,980 alloy atoms 114 + 153 us at one lane
// with the general powers, 20 + 23 us so with the table's straight products.
// A batch keeps one size-independent default, so that a walker gives the same
// bits alone and among others.
}  // namespace
void akmc_single_variant(int n, int &lpa, int &unroll)
{
    lpa = n < 16384 ? 64 : 8;
    unroll = n < 16384 ? 1 : 2;
}
namespace {

bool orthorhombic(const double *lat)
{
    return lat[1] == 0.0 && lat[2] == 0.0 && lat[3] == 0.0 && lat[5] == 0.0 && lat[6] == 0.0 && lat[7] == 0.0 &&
           lat[0] > 0 && lat[4] > 0 && lat[8] > 0;
}

// eta and reciprocal shells from the Madelung accuracy
// (potentials/pair/Field.cpp:129-132, Ewald.cpp:88-120) for an orthorhombic cell
void ewald_params(const akmc_field_s *f, const double *L, double &eta, int g[3])
{
    if (f->explicit_ewald) {
        eta = f->eta;
        for (int a = 0; a < 3; ++a) g[a] = f->gcell[a];
        return;
    }
    double eps = std::fmin(std::fabs(f->madelung_acc), 0.5);
    double tol = std::sqrt(std::fabs(std::log(eps * f->rc)));
    eta = std::sqrt(std::fabs(std::log(eps * f->rc * tol))) / f->rc;
    double tol1 = std::sqrt(-std::log(eps * f->rc * std::pow(2.0 * tol * eta, 2)));
    for (int a = 0; a < 3; ++a) g[a] = (int)std::rint(0.25 + L[a] * eta * tol1 / kPI);
}

// half-space k set (Ewald.cpp:188-319) for an orthorhombic cell; rcpcut is
// min_a g_a / L_a
void kvectors(const akmc_field_s *f, const double *L, double eta, const int g[3], std::vector<int> &kn,
              std::vector<double> &kv, std::vector<double> &g0, std::vector<double> &g1)
{
    double cut = std::min({g[0] / L[0], g[1] / L[1], g[2] / L[2]});
    double cut2 = cut * cut, vol = L[0] * L[1] * L[2];
    double etasq = eta * eta, gsqfct = 1.0 / (4.0 * etasq);
    double gfct0 = kCTOEV * kPI / (etasq * vol), gfct1 = gsqfct * gfct0;
    for (int nx = 0; nx <= g[0]; ++nx)
        for (int ny = -g[1]; ny <= g[1]; ++ny)
            for (int nz = -g[2]; nz <= g[2]; ++nz) {
                double x = nx / L[0], y = ny / L[1], z = nz / L[2];
                double gsq = x * x + y * y + z * z;
                if (gsq < cut2 && gsq > 1.0e-8) {
                    double kx = 2.0 * kPI * x, ky = 2.0 * kPI * y, kz = 2.0 * kPI * z;
                    double ksq = kx * kx + ky * ky + kz * kz, xg = ksq * gsqfct;
                    double gzz = std::exp(-xg) / xg;
                    kn.push_back(nx);
                    kn.push_back(ny);
                    kn.push_back(nz);
                    kv.push_back(kx);
                    kv.push_back(ky);
                    kv.push_back(kz);
                    g0.push_back(kx < 1.0e-8 ? gzz * gfct0 : gzz * gfct0 * 2.0);
                    g1.push_back(-2.0 * gzz * (1.0 + 1.0 / xg) * gfct1);
                }
            }
    (void)f;
}

int check_cell(const akmc_field_s *f, const double *lat)
{
    if (!orthorhombic(lat)) return fail(AKMC_EUNSUPPORTED, "only orthorhombic cells are supported on the device");
    if (f->rc < 1.0) return fail(AKMC_EINVAL, "short range cutoff is too small : %g", f->rc);
    double mind = std::min({lat[0], lat[4], lat[8]});
    // image-convention checks: metal Field.cpp:53-60, pair Field.cpp:99-106
    double radius = f->kind == 0 ? (f->nbrlist ? f->rc + f->verlet_shell : f->rc) : f->rc + f->verlet_shell;
    if (f->min_image && radius > mind / 2)
        return fail(AKMC_EINVAL, "short range cutoff too large for simulation box: cutoff %g minimum dimension %g",
                    f->rc, mind);
    return AKMC_SUCCESS;
}

template <typename T>
int dalloc(akmc_batch_t b, T **p, size_t n)
{
    if (n == 0) n = 1;
    HIPCHK(hipMalloc((void **)p, n * sizeof(T)));
    b->allocs.push_back((void *)*p);
    return AKMC_SUCCESS;
}

#define TRY(expr)                      \
    do {                               \
        int rc_ = (expr);              \
        if (rc_ != AKMC_SUCCESS) return rc_; \
    } while (0)

// device copy of the EAM tables (once per field) and their addresses in the
// host FieldDev (again after every build_tables)
int ensure_eam_tables(akmc_field_t f)
{
    if (f->eam.empty()) return AKMC_SUCCESS;
    std::vector<size_t> off_d, off_p, off_e;
    size_t total = 0;
    for (const EamPot &e : f->eam) {
        off_d.push_back(total);
        total += e.nr;
        off_p.push_back(total);
        total += 3 * (size_t)e.nr;
        off_e.push_back(total);
        total += 2 * (size_t)e.nrho;
    }
    if (!f->eam_dev) {
        // value tables as (t_i, t_{i+1} - t_i); derivative tables are the
        // forward differences (MetalPotential.cpp:388-392), last entry 0
        auto deriv = [](const std::vector<double> &t, double h) {
            std::vector<double> d(t.size(), 0.0);
            for (size_t i = 0; i + 1 < t.size(); ++i) d[i] = (t[i + 1] - t[i]) / h;
            return d;
        };
        auto pairs = [](const std::vector<double> &t, size_t i) {
            return make_double2(t[i], i + 1 < t.size() ? t[i + 1] - t[i] : 0.0);
        };
        std::vector<double2> h(total);
        for (size_t k = 0; k < f->eam.size(); ++k) {
            const EamPot &e = f->eam[k];
            const std::vector<double> dphi = deriv(e.phi, e.dr), drho = deriv(e.rho, e.dr), dF = deriv(e.F, e.drho);
            for (int i = 0; i < e.nr; ++i) {
                h[off_d[k] + i] = pairs(e.rho, i);
                h[off_p[k] + 3 * (size_t)i + 0] = pairs(e.phi, i);
                h[off_p[k] + 3 * (size_t)i + 1] = pairs(dphi, i);
                h[off_p[k] + 3 * (size_t)i + 2] = pairs(drho, i);
            }
            for (int i = 0; i < e.nrho; ++i) {
                h[off_e[k] + 2 * (size_t)i + 0] = pairs(e.F, i);
                h[off_e[k] + 2 * (size_t)i + 1] = pairs(dF, i);
            }
        }
        HIPCHK(hipMalloc((void **)&f->eam_dev, total * sizeof(double2)));
        HIPCHK(hipMemcpy(f->eam_dev, h.data(), total * sizeof(double2), hipMemcpyHostToDevice));
    }
    for (size_t k = 0; k < f->eam.size(); ++k) {
        f->host.eamt[k].dens = f->eam_dev + off_d[k];
        f->host.eamt[k].pair = f->eam_dev + off_p[k];
        f->host.eamt[k].emb = f->eam_dev + off_e[k];
    }
    return AKMC_SUCCESS;
}

// the erfc mesh of the damped-shifted Coulomb sum, Field::fieldErfcGen
// (potentials/pair/Field.cpp:19-73): erfc(alpha r)/r by Abramowitz and
// Stegun 7.1.26 and (that + 2 alpha/sqrt(pi) exp(-alpha^2 r^2)) / r^2 at
// r = i rc / (n - 4); the shift terms are the values at rc.  The
// reference's point count (MAXMESH) lives in its missing Constants.h; the
// count here is this library's choice.
constexpr int kDsfMesh = 5000;

int ensure_dsf_mesh(akmc_field_t f)
{
    if (f->kind != 1 || f->do_ewald != 2) return AKMC_SUCCESS;
    const int n = kDsfMesh;
    const double rc = f->rc, a = f->dsf_alpha, del = rc / (n - 4);
    std::vector<double> h(2 * (size_t)n, 0.0);
    const double a1 = 0.254829592, a2 = -0.284496736, a3 = 1.421413741, a4 = -1.453152027, a5 = 1.061405429,
                 pp = 0.3275911;
    for (int i = 1; i < n; ++i) {
        const double r = (double)i * del, rsq = r * r;
        const double tt = 1.0 / (1.0 + pp * a * r);
        const double ex = std::exp(-std::pow(a * r, 2.0));
        h[i] = tt * (a1 + tt * (a2 + tt * (a3 + tt * (a4 + tt * a5)))) * ex / r;
        h[n + i] = (h[i] + 2.0 * (a / 1.7724538509055159) * ex) / rsq;
    }
    if (!f->dsf_dev) {
        HIPCHK(hipMalloc((void **)&f->dsf_dev, 2 * (size_t)n * sizeof(double)));
        HIPCHK(hipMemcpy(f->dsf_dev, h.data(), 2 * (size_t)n * sizeof(double), hipMemcpyHostToDevice));
    }
    FieldDev &d = f->host;
    d.dsf_e = f->dsf_dev;
    d.dsf_f = f->dsf_dev + n;
    d.dsf_n = n;
    d.dsf_del = del;
    d.dsf_rfld0 = h[n - 4];
    d.dsf_rfld1 = rc * h[n + n - 4];
    d.eta = a;
    return AKMC_SUCCESS;
}

int batch_build(akmc_field_t f, int W, const int *natoms, const double *lat, akmc_batch_t b)
{
    b->f = f;
    b->W = W;
    b->hw.resize(W);
    int A = 0, ncells = 0, G1 = 1, maxnk = 0;
    double rl = f->rc + f->skin;
    double max_density = 0.0;
    for (int w = 0; w < W; ++w) {
        const double *lw = lat + 9 * w;
        TRY(check_cell(f, lw));
        if (natoms[w] <= 0 || natoms[w] > AKMC_MAX_WALKER_ATOMS)
            return fail(AKMC_EINVAL, "walker %d: atom count %d out of range", w, natoms[w]);
        WalkerDev &h = b->hw[w];
        std::memset(&h, 0, sizeof h);
        h.off = A;
        h.n = natoms[w];
        A += h.n;
        h.L[0] = lw[0];
        h.L[1] = lw[4];
        h.L[2] = lw[8];
        for (int a = 0; a < 3; ++a) {
            h.invL[a] = 1.0 / h.L[a];
            h.nc[a] = std::min(AKMC_MAX_CELLS_AXIS, std::max(1, (int)std::floor(h.L[a] / rl)));
            h.shells[a] = (int)(rl / h.L[a]) + 1;
            if (h.shells[a] > 7) return fail(AKMC_ECAPACITY, "walker %d: more than 7 image shells", w);
        }
        h.cell_off = ncells;
        ncells += h.nc[0] * h.nc[1] * h.nc[2];
        max_density = std::max(max_density, h.n / (h.L[0] * h.L[1] * h.L[2]));
        max_density = std::max(max_density, f->list_density);
        if (f->kind == 1 && f->do_ewald == 1) {
            double eta;
            int g[3];
            ewald_params(f, h.L, eta, g);
            f->host.eta = eta;
            std::vector<int> kn;
            std::vector<double> kv, g0, g1;
            kvectors(f, h.L, eta, g, kn, kv, g0, g1);
            h.k_off = (int)b->hg0.size();
            h.nk = (int)g0.size();
            h.gmax = std::max({g[0], g[1], g[2]});
            G1 = std::max(G1, h.gmax + 1);
            maxnk = std::max(maxnk, h.nk);
            b->hk_n.insert(b->hk_n.end(), kn.begin(), kn.end());
            b->hk_v.insert(b->hk_v.end(), kv.begin(), kv.end());
            b->hg0.insert(b->hg0.end(), g0.begin(), g0.end());
            b->hg1.insert(b->hg1.end(), g1.begin(), g1.end());
            f->nk_last = h.nk;
        }
    }
    b->A = A;
    int nk = (int)b->hg0.size();
    // neighbour capacity: 1.6x the expected count in the list sphere + 64
    double expect = 4.0 / 3.0 * kPI * rl * rl * rl * max_density;
    int maxnb = ((int)(1.6 * expect) + 64 + 31) / 32 * 32;
    // list offsets are 32-bit row A + i products (24-bit operands)
    if (A >= (1 << 24) || (size_t)(maxnb + AKMC_NB_PAD_ROWS) * (size_t)A >= ((size_t)1 << 32))
        return fail(AKMC_ECAPACITY, "batch of %d atoms with %d list entries per atom is too large", A, maxnb);
    BatchDev &d = b->d;
    std::memset(&d, 0, sizeof d);
    d.A = A;
    d.W = W;
    d.maxnb = maxnb;
    d.lpa = 4;  // one default for every batch size (512 walkers, unstaged: 1.13 ms an evaluation, 1.80 at 1 x 1)
    d.unroll = 4;
    {
        int nmax = 0;
        for (int w = 0; w < W; ++w) nmax = std::max(nmax, natoms[w]);
        d.nb16 = (f->kind == 0 && f->min_image && nmax <= 65535) ? 1 : 0;
        // above this size a 256-thread workgroup loops 64 times over a
        // walker's atoms per vector operation of its state machine
        constexpr int kWideLogicAtoms = 16384;
        b->logic_wide = nmax >= kWideLogicAtoms;
    }
    d.ncells_total = ncells;
    d.nk_total = nk;
    d.G1 = G1;
    d.maxnk = maxnk;
    d.maxn = *std::max_element(natoms, natoms + W);
    HIPCHK(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
    HIPCHK(hipEventCreate(&b->ev0));
    HIPCHK(hipEventCreate(&b->ev1));
    WalkerDev *wd;
    int *wk, *tp;
    double *q;
    TRY(dalloc(b, &wd, W));
    TRY(dalloc(b, &wk, A));
    {
        const size_t a = A, w = W, flags = 24 * a + 4 * a;
        b->io_q = (flags + 8 * w + 15) / 16 * 16;
        b->io_in = b->io_q + 8 * a;
        b->io_out = (b->io_in + 255) / 256 * 256;
        b->io_end = b->io_out + 24 * a + w * sizeof(WalkerOut) + sizeof(int);
        TRY(dalloc(b, &b->io, b->io_end));
        d.x = (double *)b->io;
        d.y = d.x + a;
        d.z = d.y + a;
        tp = (int *)(d.z + a);
        d.rebuild = tp + a;
        d.active = d.rebuild + w;
        q = (double *)(b->io + b->io_q);
        d.fx = (double *)(b->io + b->io_out);
        d.fy = d.fx + a;
        d.fz = d.fy + a;
        d.out = (WalkerOut *)(d.fz + a);
        d.overflow = (int *)(d.out + w);
    }
    d.walkers = wd;
    d.wk = wk;
    d.type = tp;
    d.q = q;
    TRY(dalloc(b, &d.p4, A));
    TRY(dalloc(b, &d.xr, A));
    TRY(dalloc(b, &d.yr, A));
    TRY(dalloc(b, &d.zr, A));
    TRY(dalloc(b, &d.nbr, (size_t)(maxnb + AKMC_NB_PAD_ROWS) * A));
    TRY(dalloc(b, &d.nnb, A));
    TRY(dalloc(b, &d.nnear, A));
    TRY(dalloc(b, &d.cell_count, ncells));
    TRY(dalloc(b, &d.cell_start, ncells));
    TRY(dalloc(b, &d.cell_atoms, A));
    TRY(dalloc(b, &d.rho, A));
    TRY(dalloc(b, &d.inv_sqrt_rho, A));
    TRY(dalloc(b, &d.isr64, A));
    TRY(dalloc(b, &d.e_a, A));
    TRY(dalloc(b, &d.e_b, A));
    TRY(dalloc(b, &d.e_a64, A));
    TRY(dalloc(b, &d.e_b64, A));
    TRY(dalloc(b, &d.e_c, A));
    TRY(dalloc(b, &d.st_atom, (size_t)6 * A));
    if (nk > 0) {
        int *kn;
        double *kv, *g0, *g1;
        TRY(dalloc(b, &kn, (size_t)3 * nk));
        TRY(dalloc(b, &kv, (size_t)3 * nk));
        TRY(dalloc(b, &g0, nk));
        TRY(dalloc(b, &g1, nk));
        // transpose to [3][nk]
        std::vector<int> tn(3 * (size_t)nk);
        std::vector<double> tv(3 * (size_t)nk);
        for (int k = 0; k < nk; ++k)
            for (int a = 0; a < 3; ++a) {
                tn[(size_t)a * nk + k] = b->hk_n[3 * (size_t)k + a];
                tv[(size_t)a * nk + k] = b->hk_v[3 * (size_t)k + a];
            }
        HIPCHK(hipMemcpy(kn, tn.data(), tn.size() * sizeof(int), hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(kv, tv.data(), tv.size() * sizeof(double), hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(g0, b->hg0.data(), nk * sizeof(double), hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(g1, b->hg1.data(), nk * sizeof(double), hipMemcpyHostToDevice));
        d.kn = kn;
        d.kv = kv;
        d.g0 = g0;
        d.g1 = g1;
        TRY(dalloc(b, &d.ptab, (size_t)A * 3 * G1));
        TRY(dalloc(b, &d.Ck, nk));
        TRY(dalloc(b, &d.Sk, nk));
    }
    std::vector<int> hwk(A);
    for (int w = 0; w < W; ++w)
        for (int i = 0; i < b->hw[w].n; ++i) hwk[b->hw[w].off + i] = w;
    HIPCHK(hipMemcpy(wd, b->hw.data(), W * sizeof(WalkerDev), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(wk, hwk.data(), A * sizeof(int), hipMemcpyHostToDevice));
    {
        // LDS staging: a walker's packed gather records (32 bytes per atom)
        // next to the static pair table of the multi-species kernels
        int nmax = 0, dev = 0, maxlds = 0;
        for (int w = 0; w < W; ++w) nmax = std::max(nmax, b->hw[w].n);
        HIPCHK(hipGetDevice(&dev));
        HIPCHK(hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
        const size_t bytes = (size_t)nmax * sizeof(double4);
        b->stage_ok = f->kind == 0 && bytes + sizeof(SCPairDev) * AKMC_MAXPAIR <= (size_t)maxlds;
        d.stage_bytes = (int)bytes;
        for (int li = 0; li < 4; ++li) {
            const int apc = AKMC_STAGE_BLOCK >> li;  // atoms per chunk at 1, 2, 4, 8 lanes per atom
            std::vector<int2> ch;
            for (int w = 0; w < W; ++w)
                for (int a0 = 0; a0 < b->hw[w].n; a0 += apc) ch.push_back(make_int2(w, a0));
            int2 *dc;
            TRY(dalloc(b, &dc, ch.size()));
            HIPCHK(hipMemcpy(dc, ch.data(), ch.size() * sizeof(int2), hipMemcpyHostToDevice));
            d.chunk_tab[li] = dc;
            d.nchunk_tab[li] = (int)ch.size();
        }
    }
    if (f->min_image) {
        std::vector<int2> seg;
        std::vector<int4> lw;
        for (int w = 0; w < W; ++w) {
            if (natoms[w] <= AKMC_BIN_ATOMS) continue;
            const int s0 = (int)seg.size();
            for (int a0 = 0; a0 < natoms[w]; a0 += 1024) seg.push_back(make_int2(w, a0));
            lw.push_back(make_int4(w, s0, (int)seg.size() - s0, 0));
        }
        if (!seg.empty()) {
            int2 *ds;
            int4 *dw;
            TRY(dalloc(b, &ds, seg.size()));
            TRY(dalloc(b, &dw, lw.size()));
            TRY(dalloc(b, &d.bin_cnt, seg.size() * AKMC_MAX_WALKER_CELLS));
            TRY(dalloc(b, &d.bin_cell, A));
            HIPCHK(hipMemcpy(ds, seg.data(), seg.size() * sizeof(int2), hipMemcpyHostToDevice));
            HIPCHK(hipMemcpy(dw, lw.data(), lw.size() * sizeof(int4), hipMemcpyHostToDevice));
            d.bin_seg = ds;
            d.bin_walker = dw;
            d.nbin_seg = (int)seg.size();
            d.nbin_walker = (int)lw.size();
        }
    }
    {
        std::vector<int> hcw(ncells);
        for (int w = 0; w < W; ++w) {
            const WalkerDev &h = b->hw[w];
            for (int c = 0; c < h.nc[0] * h.nc[1] * h.nc[2]; ++c) hcw[h.cell_off + c] = w;
        }
        int *cw;
        TRY(dalloc(b, &cw, ncells));
        HIPCHK(hipMemcpy(cw, hcw.data(), ncells * sizeof(int), hipMemcpyHostToDevice));
        d.cell_wk = cw;
        TRY(dalloc(b, &d.cell_work, (size_t)ncells + A / 16 + 1));  // list-build items (cell, home chunk)
        TRY(dalloc(b, &d.cell_work_n, 1));
        HIPCHK(hipMemset(d.cell_work_n, 0, sizeof(int)));
    }
    HIPCHK(hipMemset(d.rebuild, 0, W * sizeof(int)));
    {
        std::vector<int> one(W, f->fp64 ? 2 : 1);
        HIPCHK(hipMemcpy(d.active, one.data(), W * sizeof(int), hipMemcpyHostToDevice));
    }
    HIPCHK(hipMemset(d.overflow, 0, sizeof(int)));
    HIPCHK(hipMemset(d.e_c, 0, A * sizeof(double)));
    HIPCHK(hipMemset((void *)d.q, 0, A * sizeof(double)));
    // device copy of the field (the eta of the last walker; all walkers of a
    // batch share the field's eta rule)
    if (!f->dev) HIPCHK(hipMalloc(&f->dev, sizeof(FieldDev)));
    TRY(ensure_eam_tables(f));
    TRY(ensure_dsf_mesh(f));
    HIPCHK(hipMemcpy(f->dev, &f->host, sizeof(FieldDev), hipMemcpyHostToDevice));
    d.field = f->dev;
    b->hout.resize(W);
    unsigned long long *cnt = akmc_rebuild_counter_ptr();
    if (!cnt) return fail(AKMC_EHIP, "rebuild counter allocation failed");
    d.rebuild_count = cnt;
    HIPCHK(hipMemcpy(&b->rebuild_base, cnt, sizeof b->rebuild_base, hipMemcpyDeviceToHost));
    return AKMC_SUCCESS;
}

void batch_free(akmc_batch_t b)
{
    if (!b) return;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    for (void *p : b->allocs) (void)hipFree(p);
    if (b->ev0) (void)hipEventDestroy(b->ev0);
    for (auto &e : b->evp)
        if (e) (void)hipEventDestroy(e);
    if (b->ev1) (void)hipEventDestroy(b->ev1);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    for (auto &row : b->kev)
        for (auto &e : row)
            if (e) (void)hipEventDestroy(e);
    if (b->hws_pin) (void)hipHostFree(b->hws_pin);
    if (b->ov_pin) (void)hipHostFree(b->ov_pin);
    if (b->zf_pin) (void)hipHostFree(b->zf_pin);
    if (b->gat_pin) (void)hipHostFree(b->gat_pin);
    if (b->gat_dev) (void)hipFree(b->gat_dev);
    if (b->desc_dev) (void)hipFree(b->desc_dev);
    if (b->io_pin) (void)hipHostFree(b->io_pin);
    if (b->stage_pin) (void)hipHostFree(b->stage_pin);
    if (b->stage_dev) (void)hipFree(b->stage_dev);
    if (b->st_pin) (void)hipHostFree(b->st_pin);
    if (b->stage_ev) (void)hipEventDestroy(b->stage_ev);
    if (b->st_ev) (void)hipEventDestroy(b->st_ev);
    if (b->side) (void)hipStreamDestroy(b->side);
    for (double *p : b->hv_pin)
        if (p) (void)hipHostFree(p);
    delete b;
}

int batch_mode(akmc_batch_t b) { return b->f->fp64 ? 2 : 1; }

int run_forces(akmc_batch_t b, int want_stress)
{
    akmc_launch_forces_impl(b->d, b->f->host, batch_mode(b), want_stress, b->stream);
    HIPCHK(hipGetLastError());
    return AKMC_SUCCESS;
}

// the error of a nonzero overflow word
int overflow_error(akmc_batch_t b, int ov)
{
    if (ov & AKMC_OV_LIST) return fail(AKMC_ECAPACITY, "neighbour list capacity %d exceeded", b->d.maxnb);
    if (ov & AKMC_OV_EAM_RHO) return fail(AKMC_EINVAL, "the rho for embedding is out of bounds of its EAM table");
    return AKMC_SUCCESS;
}

int check_overflow(akmc_batch_t b)
{
    int ov = 0;
    HIPCHK(hipMemcpyAsync(&ov, b->d.overflow, sizeof(int), hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return overflow_error(b, ov);
}

// forces, energy records and the overflow flag of a small batch in one
// transfer (into hout and the pinned buffer)
int fetch_all(akmc_batch_t b)
{
    char *pin = b->io_pin + b->io_out;
    HIPCHK(hipMemcpyAsync(pin, b->io + b->io_out, b->io_end - b->io_out, hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    const char *out = pin + 24 * (size_t)b->A;
    std::memcpy((void *)b->hout.data(), out, b->W * sizeof(WalkerOut));
    int ov;
    std::memcpy(&ov, out + b->W * sizeof(WalkerOut), sizeof ov);
    return overflow_error(b, ov);
}

int fetch_out(akmc_batch_t b)
{
    HIPCHK(hipMemcpyAsync(b->hout.data(), b->d.out, b->W * sizeof(WalkerOut), hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return AKMC_SUCCESS;
}

void to_energy(const WalkerOut &o, akmc_energy *e)
{
    e->total = o.total;
    e->rcp = o.rcp;
    e->real = o.real;
    e->many = o.many;
    e->vdw = o.vdw;
    e->ext = 0.0;
}

// in-place wraps of the caller's arrays, as Field::calculateForces does
// (potentials/metal/Field.cpp:1855-1920)
void host_wrap(bool min_image, const double *lat, int n, double *x, double *y, double *z)
{
    double L[3] = {lat[0], lat[4], lat[8]};
    for (int i = 0; i < n; ++i) {
        double s[3] = {x[i] / L[0], y[i] / L[1], z[i] / L[2]};
        for (int a = 0; a < 3; ++a) {
            if (min_image) {
                s[a] -= std::rint(s[a]);
            } else {
                if (s[a] < 0.0) s[a] += 1.0;
                if (s[a] >= 1.0) s[a] -= 1.0;
            }
        }
        x[i] = s[0] * L[0];
        y[i] = s[1] * L[1];
        z[i] = s[2] * L[2];
    }
}

// up to this much goes through pinned memory: a 255-atom call is seven
// pageable copies of 5-15 us otherwise; past it a pageable copy streams as
// fast as the host can fill a pinned buffer
constexpr size_t kPinnedIo = (size_t)4 << 20;

// the batch's force calls move their data through its pinned buffer
bool pinned_io(akmc_batch_t b) { return b->io_end <= kPinnedIo && !b->search_alloc; }

int ensure_io_pin(akmc_batch_t b)
{
    if (b->io_pin && b->io_pin_n >= b->io_end) return AKMC_SUCCESS;
    if (b->io_pin) HIPCHK(hipHostFree(b->io_pin));
    b->io_pin = nullptr;
    b->io_pin_n = 0;
    HIPCHK(hipHostMalloc((void **)&b->io_pin, b->io_end, hipHostMallocDefault));
    b->io_pin_n = b->io_end;
    return AKMC_SUCCESS;
}

int ensure_single(akmc_field_t f, int n, const double *lat)
{
    bool same = f->single && f->single_n == n && std::memcmp(f->single_lat, lat, sizeof f->single_lat) == 0;
    if (same) return AKMC_SUCCESS;
    // the pinned buffer (at most kPinnedIo) passes from cell to cell
    char *pin = nullptr;
    size_t pin_n = 0;
    if (f->single) {
        std::swap(pin, f->single->io_pin);
        std::swap(pin_n, f->single->io_pin_n);
        batch_free(f->single);
    }
    f->single = new akmc_batch_s();
    f->single->io_pin = pin;
    f->single->io_pin_n = pin_n;
    int rc = batch_build(f, 1, &n, lat, f->single);
    if (rc != AKMC_SUCCESS) {
        batch_free(f->single);
        f->single = nullptr;
        return rc;
    }
    akmc_single_variant(n, f->single->d.lpa, f->single->d.unroll);
    f->single_n = n;
    std::memcpy(f->single_lat, lat, sizeof f->single_lat);
    return AKMC_SUCCESS;
}

// wait: returns with the host arrays and the pinned buffer free for reuse (a
// caller that synchronises the stream itself need not)
int upload(akmc_batch_t b, const double *x, const double *y, const double *z, const int *type, const double *q,
           bool wait = true)
{
    size_t A = b->A;
    int ns = (int)b->f->species.size();
    for (size_t i = 0; i < A; ++i)
        if (type[i] < 0 || type[i] >= ns) return fail(AKMC_EINVAL, "atom %zu: species %d out of range", i, type[i]);
    if (pinned_io(b)) {
        TRY(ensure_io_pin(b));
        double *px = (double *)b->io_pin;
        std::memcpy(px, x, A * sizeof(double));
        std::memcpy(px + A, y, A * sizeof(double));
        std::memcpy(px + 2 * A, z, A * sizeof(double));
        int *pt = (int *)(px + 3 * A);
        std::memcpy(pt, type, A * sizeof(int));
        std::fill(pt + A, pt + A + b->W, 1);                           // fresh lists
        std::fill(pt + A + b->W, pt + A + 2 * b->W, batch_mode(b));  // every walker is evaluated
        if (q) std::memcpy(b->io_pin + b->io_q, q, A * sizeof(double));
        HIPCHK(hipMemcpyAsync(b->io, b->io_pin, q ? b->io_in : b->io_q, hipMemcpyHostToDevice, b->stream));
        if (wait) HIPCHK(hipStreamSynchronize(b->stream));
        return AKMC_SUCCESS;
    }
    HIPCHK(hipMemcpyAsync(b->d.x, x, A * sizeof(double), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(b->d.y, y, A * sizeof(double), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(b->d.z, z, A * sizeof(double), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync((void *)b->d.type, type, A * sizeof(int), hipMemcpyHostToDevice, b->stream));
    if (q) HIPCHK(hipMemcpyAsync((void *)b->d.q, q, A * sizeof(double), hipMemcpyHostToDevice, b->stream));
    // a fresh configuration always gets fresh lists, and every walker is
    // evaluated by plain force calls
    std::vector<int> ones(b->W, 1), mode(b->W, batch_mode(b));
    HIPCHK(hipMemcpyAsync(b->d.rebuild, ones.data(), b->W * sizeof(int), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(b->d.active, mode.data(), b->W * sizeof(int), hipMemcpyHostToDevice, b->stream));
    // a running search's zone does not survive new positions; neither do the
    // resident kernel's lists, so its walkers go on through the chain
    if (b->zflag) HIPCHK(hipMemsetAsync(b->zflag, 0, b->W * sizeof(int), b->stream));
    if (b->search_alloc) {
        HIPCHK(hipMemcpyAsync(b->s.X, x, A * sizeof(double), hipMemcpyHostToDevice, b->stream));
        HIPCHK(hipMemcpyAsync(b->s.X + A, y, A * sizeof(double), hipMemcpyHostToDevice, b->stream));
        HIPCHK(hipMemcpyAsync(b->s.X + 2 * A, z, A * sizeof(double), hipMemcpyHostToDevice, b->stream));
    }
    HIPCHK(hipStreamSynchronize(b->stream));
    if (b->search_alloc)
        for (int w = 0; w < b->W; ++w) b->hzflag[w] = b->zf_pin[w] = 0;
    return AKMC_SUCCESS;
}


// f(first atom, atoms) for each run of neighbouring selected walkers (all
// when null): their slices lie together, so a run is one transfer (one per
// walker took 30 ms for 512)
template <typename F>
int for_runs(akmc_batch_t b, const int *walkers, F f)
{
    for (int w = 0; w < b->W;) {
        if (walkers && !walkers[w]) {
            ++w;
            continue;
        }
        const int off = b->hw[w].off;
        int end = off;
        for (; w < b->W && (!walkers || walkers[w]); ++w) end = b->hw[w].off + b->hw[w].n;
        TRY(f((size_t)off, (size_t)(end - off)));
    }
    return AKMC_SUCCESS;
}

// rebuild the free-atom lists of the selected walkers (all when null) from
// the host copy of the frozen mask and upload them
int upload_active(akmc_batch_t b, const int *walkers)
{
    for (int w = 0; w < b->W; ++w) {
        if (walkers && !walkers[w]) continue;
        const int off = b->hw[w].off, n = b->hw[w].n;
        int m = 0;
        for (int i = 0; i < n; ++i)
            if (!b->hfrozen[off + i]) b->hact[off + m++] = off + i;
        b->hnact[w] = m;
    }
    TRY(for_runs(b, walkers, [&](size_t off, size_t n) {
        HIPCHK(hipMemcpyAsync((void *)(b->s.act + off), b->hact.data() + off, n * sizeof(int), hipMemcpyHostToDevice,
                              b->stream));
        return (int)AKMC_SUCCESS;
    }));
    HIPCHK(hipMemcpyAsync((void *)b->s.nact, b->hnact.data(), b->W * sizeof(int), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return AKMC_SUCCESS;
}

int search_alloc(akmc_batch_t b)
{
    if (b->search_alloc) return AKMC_SUCCESS;
    size_t A3 = 3 * (size_t)b->A;
    TRY(dalloc(b, &b->s.X, A3));
    TRY(dalloc(b, &b->s.N, A3));
    TRY(dalloc(b, &b->s.V, A3));
    TRY(dalloc(b, &b->s.F0, A3));
    TRY(dalloc(b, &b->s.F1, A3));
    TRY(dalloc(b, &b->s.T, A3));
    int *fr;
    TRY(dalloc(b, &fr, b->A));
    HIPCHK(hipMemset(fr, 0, b->A * sizeof(int)));
    b->s.frozen = fr;
    int *act, *nact;
    TRY(dalloc(b, &act, b->A));
    TRY(dalloc(b, &nact, b->W));
    TRY(dalloc(b, &b->s.evals32, b->W));
    HIPCHK(hipMemset(b->s.evals32, 0, b->W * sizeof(unsigned long long)));
    b->s.act = act;
    b->s.nact = nact;
    b->hfrozen.assign(b->A, 0);
    b->hact.assign(b->A, 0);
    b->hnact.assign(b->W, 0);
    TRY(dalloc(b, &b->s.ws, b->W));
    HIPCHK(hipMemset(b->s.ws, 0, b->W * sizeof(WalkerState)));
    TRY(dalloc(b, &b->zflag, b->W));
    TRY(dalloc(b, &b->zmark, b->A));
    TRY(dalloc(b, &b->zlist, b->A));
    TRY(dalloc(b, &b->nz, b->W));
    // a list chunk holds at least 32 slots (256 threads at 8 lanes per atom)
    for (int k = 0; k < 4; ++k) TRY(dalloc(b, &b->wl_tab[k], (size_t)b->A / 32 + b->W + 1));
    TRY(dalloc(b, &b->wl_count, 4));
    HIPCHK(hipMemset(b->wl_count, 0, 4 * sizeof(int)));
    {
        // persistent grids: every CU, as many staged workgroups as its 160 KB
        // of LDS holds (at most 2), 8 plain ones; multiples of the 8 XCDs
        int dev = 0, ncu = 0;
        HIPCHK(hipGetDevice(&dev));
        HIPCHK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
        const size_t lds = (size_t)b->d.stage_bytes + sizeof(SCPairDev) * AKMC_MAXPAIR;
        const int res = std::max(1, std::min(2, (int)(163840 / std::max<size_t>(lds, 1))));
        b->wl_grid_staged = ((ncu * res + 7) / 8) * 8;
        b->wl_grid_plain = ((ncu * 8 + 7) / 8) * 8;
    }
    HIPCHK(hipMemset(b->zflag, 0, b->W * sizeof(int)));
    HIPCHK(hipMemset(b->nz, 0, b->W * sizeof(int)));
    b->hzflag.assign(b->W, 0);
    // X starts at the resident positions
    size_t A = b->A;
    HIPCHK(hipMemcpy(b->s.X, b->d.x, A * sizeof(double), hipMemcpyDeviceToDevice));
    HIPCHK(hipMemcpy(b->s.X + A, b->d.y, A * sizeof(double), hipMemcpyDeviceToDevice));
    HIPCHK(hipMemcpy(b->s.X + 2 * A, b->d.z, A * sizeof(double), hipMemcpyDeviceToDevice));
    b->hws.assign(b->W, WalkerState{});
    TRY(upload_active(b, nullptr));
    HIPCHK(hipHostMalloc((void **)&b->hws_pin, b->W * sizeof(WalkerState), hipHostMallocDefault));
    HIPCHK(hipHostMalloc((void **)&b->ov_pin, sizeof(int), hipHostMallocDefault));
    HIPCHK(hipHostMalloc((void **)&b->zf_pin, b->W * sizeof(int), hipHostMallocDefault));
    std::fill(b->zf_pin, b->zf_pin + b->W, 0);
    HIPCHK(hipHostMalloc((void **)&b->st_pin, b->W * sizeof(StartItem), hipHostMallocDefault));
    TRY(dalloc(b, &b->st_dev, b->W));
    HIPCHK(hipEventCreateWithFlags(&b->stage_ev, hipEventDisableTiming));
    HIPCHK(hipEventCreateWithFlags(&b->st_ev, hipEventDisableTiming));
    b->search_alloc = true;
    return AKMC_SUCCESS;
}

void drop_graph(akmc_batch_t b)
{
    if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->gexec = nullptr;
    b->graph = nullptr;
    b->graph_steps = 0;
}

// active zones apply to minimum-image Sutton-Chen fields
bool zone_usable(akmc_batch_t b)
{
    const FieldDev &h = b->f->host;
    return b->zflag && h.kind == 0 && !h.eam && h.min_image;
}

// a search of walker w runs in the resident kernel, as far as the host can
// tell: a rule on the walker and its field alone, so that its results do not
// depend on the batch it is in (the device then tries its first list build,
// k_res_admit)
bool resident_walker(akmc_batch_t b, int w)
{
    const int m = b->hnact[w], n = b->hw[w].n;
    return zone_usable(b) && b->res_on && !b->res_none && b->f->host.nspec <= 4 && m > 0 && m < n && m <= AKMC_RES_FREE &&
           n <= AKMC_RES_ATOMS;
}

// the buffers of the resident walkers; where there is no memory for them
// (some 200 KB a walker) every walker of the batch takes the chain
int ensure_resident(akmc_batch_t b)
{
    if (b->r.on || b->res_none) return AKMC_SUCCESS;
    const size_t W = b->W, A = b->A, had = b->allocs.size();
    ResidentDev r{};
    r.fcap = b->d.maxnb;
    auto alloc = [&]() {
        TRY(dalloc(b, &r.n, W));
        TRY(dalloc(b, &r.slot, W * AKMC_RES_SLOTS));
        TRY(dalloc(b, &r.mask, W * AKMC_RES_SLOTS * 4));
        TRY(dalloc(b, &r.task, W * AKMC_RES_SLOTS));
        TRY(dalloc(b, &r.fslot, W * AKMC_RES_FREE));
        TRY(dalloc(b, &r.flist, W * AKMC_RES_FREE * r.fcap));
        TRY(dalloc(b, &r.fcnt, W * AKMC_RES_FREE));
        TRY(dalloc(b, &r.ref, W * 3 * AKMC_RES_FREE));
        TRY(dalloc(b, &r.eout, W * 4));
        TRY(dalloc(b, &r.eok, W));
        for (int p = 0; p < 2; ++p) {
            TRY(dalloc(b, &r.base_rho[p], A));
            TRY(dalloc(b, &r.base_ep[p], A));
        }
        return dalloc(b, &b->res_args, 1);
    };
    if (alloc() != AKMC_SUCCESS) {
        (void)hipGetLastError();
        for (size_t k = had; k < b->allocs.size(); ++k) (void)hipFree(b->allocs[k]);
        b->allocs.resize(had);
        b->res_args = nullptr;
        b->res_none = true;
        return AKMC_SUCCESS;
    }
    r.on = 1;
    b->r = r;
    return AKMC_SUCCESS;
}

BatchDev step_dev(akmc_batch_t b);

// brings the resident kernel's descriptors up to date (in stream order: a
// chunk in flight keeps the ones it was launched with)
int sync_res_args(akmc_batch_t b)
{
    if (!b->r.on) return AKMC_SUCCESS;
    ResArgs a;
    std::memset((void *)&a, 0, sizeof a);
    a.b = step_dev(b);
    a.s = b->s;
    if (std::memcmp(&a, &b->res_host, sizeof a) == 0) return AKMC_SUCCESS;
    b->res_host = a;
    HIPCHK(hipMemcpyAsync((void *)b->res_args, &b->res_host, sizeof a, hipMemcpyHostToDevice, b->stream));
    return AKMC_SUCCESS;
}

// how the running walkers' micro-steps run: 0 the chain alone, 1 the chain
// and the resident kernel, 2 every running walker is resident
int resident_mode(akmc_batch_t b)
{
    if (!b->r.on) return 0;
    int res = 0, other = 0;
    for (int w = 0; w < b->W; ++w) {
        const WalkerState &ws = b->hws[w];
        if (ws.kind == WK_IDLE || ws.state == ST_DONE) continue;
        if (b->hzflag[w] & AKMC_ZONE_RES) ++res;
        else ++other;
    }
    return res == 0 ? 0 : other ? 1 : 2;
}

// the batch view of the search micro-steps: the plain one plus the pair
// energies in pass 1, the search variants and the zones
BatchDev step_dev(akmc_batch_t b)
{
    BatchDev d = b->d;
    const FieldDev &h = b->f->host;
    if (h.kind == 0 && !h.eam && h.min_image) {
        d.pe1 = 1;
        for (int k = 0; k < 4; ++k) d.wl_tab[k] = b->wl_tab[k];
        d.wl_count = b->wl_count;
        d.wl_grid_staged = b->wl_grid_staged;
        d.wl_grid_plain = b->wl_grid_plain;
        if (b->sv[0]) {
            d.lpa = b->sv[0];
            d.unroll = b->sv[1];
            d.staged = b->sv[2];
        }
        if (b->sv[3]) {
            d.lpa2 = b->sv[3];
            d.unroll2 = b->sv[4];
            d.staged2 = b->sv[5];
        }
        if (b->sv[6]) {
            d.lpa64 = b->sv[6];
            d.unroll64 = b->sv[7];
            d.staged64 = b->sv[8];
        }
    }
    if (zone_usable(b) && (b->zone_on || b->r.on)) {
        d.zone_off = b->zone_on ? 0 : 1;
        d.r = b->r;
        d.zfrozen = b->s.frozen;
        d.zflag = b->zflag;
        d.zmark = b->zmark;
        d.zlist = b->zlist;
        d.nz = b->nz;
        d.zact = b->s.act;
        d.znact = b->s.nact;
    }
    return d;
}

// the kernels of one force evaluation of the chain; base: with the fixed
// parts of resident walkers; sums: with the walker sums; j: the chunk's step,
// for the kernel timer's events
void enqueue_chain(akmc_batch_t b, const BatchDev &d, bool base, bool sums, int j)
{
    // FP64 pair terms run when a walker may ask for them: verification or
    // the closing FP64 energy of a relax
    const int prec = batch_mode(b) | ((b->s.verify_nl > 0 || b->s.final64) ? 2 : 0);
    const FieldDev &hf = b->f->host;
    for (int ph = 0; ph < 2; ++ph) akmc_launch_phase(d, hf, prec, 0, ph, b->stream);
    if (base) akmc_launch_res_base(d, hf, akmc_res_precisions(b->s), b->stream);
    if (b->ktimer && (prec & 1) && hf.kind == 0) {
        (void)hipEventRecord(b->kev[0][j], b->stream);
        akmc_launch_phase(d, hf, 1, 0, 2, b->stream);
        (void)hipEventRecord(b->kev[1][j], b->stream);
        if (prec & 2) akmc_launch_phase(d, hf, 2 | 4, 0, 2, b->stream);  // FP64 part of a mixed step
    } else {
        akmc_launch_phase(d, hf, prec, 0, 2, b->stream);
    }
    if (sums) akmc_launch_phase(d, hf, prec, 0, 3, b->stream);
}

// some running walker relaxes by plain FIRE with every atom free and fits the
// relax kernel (part of SearchDev, so that a captured graph is for one answer)
bool relax_fire(akmc_batch_t b) { return b->s.fire_on != 0; }

// some running resident walker waits for its fixed parts (the host's flags
// hold every bit that the device's do)
bool parts_pending(akmc_batch_t b)
{
    const int want = akmc_res_precisions(b->s);
    for (int w = 0; w < b->W; ++w) {
        const WalkerState &ws = b->hws[w];
        if (ws.kind == WK_IDLE || ws.state == ST_DONE || !(b->hzflag[w] & AKMC_ZONE_RES)) continue;
        if ((b->hzflag[w] & want) || (ws.res & AKMC_RES_WAITS)) return true;
    }
    return false;
}

// what a chunk's kernels depend on beside the descriptors
struct ChunkPlan {
    int res;       // resident_mode
    bool service;  // parts_pending
};

// The kernels of a chunk of micro-steps.  A resident walker needs the chain
// once, on its first micro-step, and a walker starts between chunks: where one
// has started, one chain evaluation serves the chunk; one resident launch takes
// all the chunk's micro-steps, and the chain goes on for the other walkers
// alone.  With zones off the chain evaluates every atom on every step; the
// kernel timer times a chain launch of every step.
void enqueue_steps(akmc_batch_t b, int steps, const ChunkPlan &p)
{
    const BatchDev d = step_dev(b);
    const bool fire = relax_fire(b), every = !b->zone_on || b->ktimer;
    const int chain = p.res < 2 || every ? steps : p.service ? 1 : 0;
    for (int j = 0; j < steps; ++j) {
        if (j < chain) enqueue_chain(b, d, p.res && j == 0 && p.service, p.res < 2, j);
        // walkers of tens of thousands of atoms: 1024-thread state machines
        if (p.res < 2) {
            if (fire) akmc_launch_relax_fire(d, b->s, b->stream);
            if (b->logic_wide) akmc_launch_search_logic_wide(d, b->s, b->stream);
            else akmc_launch_search_logic(d, b->s, b->stream);
        }
        if (p.res && (j == 0 || every))
            akmc_launch_search_resident(b->W, b->f->host, b->res_args, every ? 1 : steps, 1, j == 0 && p.service,
                                        b->stream);
    }
}

int fetch_states(akmc_batch_t b)
{
    HIPCHK(hipMemcpyAsync(b->hws.data(), b->s.ws, b->W * sizeof(WalkerState), hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return AKMC_SUCCESS;
}

// mark walkers that are done (or idle) inactive so the force kernels skip them
int refresh_active(akmc_batch_t b, int *n_running)
{
    std::vector<int> act(b->W);
    int run = 0;
    for (int w = 0; w < b->W; ++w) {
        const WalkerState &ws = b->hws[w];
        const bool fp64 = ws.kind == WK_VERIFY || ws.state == ST_R_E64;
        act[w] = (ws.kind != WK_IDLE && ws.state != ST_DONE) ? (fp64 ? 2 : batch_mode(b)) : 0;
        run += act[w];
    }
    HIPCHK(hipMemcpyAsync(b->d.active, act.data(), b->W * sizeof(int), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    *n_running = run;
    return AKMC_SUCCESS;
}

// the host may rewrite a pinned staging buffer once its last transfer,
// recorded on ev, is done
int wait_staging(hipEvent_t ev, bool &pending)
{
    if (pending) HIPCHK(hipEventSynchronize(ev));
    pending = false;
    return AKMC_SUCCESS;
}

// The listed walkers' fresh states go to the device in one pinned transfer
// and one scatter kernel, with, per walker: a fresh zone when it has frozen
// atoms (membership reset, and a full evaluation first in each precision),
// a list rebuild on its first micro-step (zones on or off alike, so both
// list the same neighbours in the same order) and its active flag.  Only the
// started walkers' device state is written, so a start may be queued behind
// a run chunk in flight (it then returns at once); otherwise it waits.
int start_walkers(akmc_batch_t b, const int *walkers, int kind, double dt0, double alpha0)
{
    TRY(wait_staging(b->st_ev, b->st_pending));
    int k = 0;
    bool resident = false;
    for (int w = 0; w < b->W; ++w) {
        if (walkers && !walkers[w]) continue;
        WalkerState ws{};
        ws.kind = kind;
        ws.state = kind == WK_RELAX ? ST_R_INIT : (kind == WK_ART ? ST_A_L0 : ST_D_F0);
        ws.it = (kind == WK_DIMER) ? 1 : 0;
        ws.status = AKMC_FAILED;
        ws.dt = dt0;
        ws.alpha = alpha0;
        // Relax.cpp:49 and ART.cpp:426 start nStep at 1
        ws.nstep = (kind == WK_RELAX || kind == WK_ART) ? 1 : 0;
        ws.inloop = 0;
        ws.verified_state = 0;
        b->hws[w] = ws;
        const int m = b->hnact[w];
        StartItem &it = b->st_pin[k++];
        it.walker = w;
        it.zflag = (m > 0 && m < b->hw[w].n) ? AKMC_ZONE_FRESH : 0;
        if (resident_walker(b, w)) TRY(ensure_resident(b));
        if (resident_walker(b, w)) {  // (not without memory)
            it.zflag |= AKMC_ZONE_RES;
            resident = true;
        }
        it.active = batch_mode(b);
        it.pad = 0;
        it.ws = ws;
        b->hzflag[w] = it.zflag;
        if (b->inflight) b->started_inflight.emplace_back(w, ws);
    }
    if (k == 0) return AKMC_SUCCESS;
    HIPCHK(hipMemcpyAsync(b->st_dev, b->st_pin, k * sizeof(StartItem), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipEventRecord(b->st_ev, b->stream));
    b->st_pending = true;
    akmc_launch_start_walkers(b->d, b->s, b->st_dev, k, b->zflag, b->hv_on ? b->harvested : nullptr,
                              b->r.on ? b->r.n : nullptr, b->stream);
    akmc_launch_probe_init(b->d, b->s, b->stream);
    if (resident) {
        TRY(sync_res_args(b));
        akmc_launch_res_admit(b->W, b->f->host, b->res_args, b->stream);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(b->zf_pin, b->zflag, b->W * sizeof(int), hipMemcpyDeviceToHost, b->stream));
    if (!b->inflight) {  // else the chunk's wait reads them
        HIPCHK(hipStreamSynchronize(b->stream));
        std::copy(b->zf_pin, b->zf_pin + b->W, b->hzflag.begin());
    }
    return AKMC_SUCCESS;
}

int ensure_lanczos(akmc_batch_t b)
{
    if (b->s.Q) return AKMC_SUCCESS;
    TRY(dalloc(b, &b->s.Q, (size_t)AKMC_LZ_MAX * 3 * b->A));
    TRY(dalloc(b, &b->s.lz, (size_t)b->W * 3 * AKMC_LZ_MAX));
    return AKMC_SUCCESS;
}

// grow a pinned host / device staging pair to n bytes
int ensure_stage(akmc_batch_t b, size_t n)
{
    if (n <= b->stage_n) return AKMC_SUCCESS;
    if (b->stage_pin) HIPCHK(hipHostFree(b->stage_pin));
    if (b->stage_dev) HIPCHK(hipFree(b->stage_dev));
    b->stage_pin = nullptr;
    b->stage_dev = nullptr;
    b->stage_n = 0;
    HIPCHK(hipHostMalloc((void **)&b->stage_pin, n, hipHostMallocDefault));
    HIPCHK(hipMalloc((void **)&b->stage_dev, n));
    b->stage_n = n;
    return AKMC_SUCCESS;
}

// per-walker start data of a saddle search: positions (optional), a
// normalised mode with frozen components removed, zero velocity, the frozen
// mask and the free-atom list.  The selected walkers' data are packed into
// one pinned buffer, copied in one transfer and scattered by one kernel.
int load_walkers(akmc_batch_t b, const int *walkers, const double *x0, const double *mode, const int *frozen)
{
    const size_t A = b->A;
    TRY(wait_staging(b->stage_ev, b->stage_pending));
    std::vector<LoadItem> items;
    size_t dwords = 0, iwords = 0, total = 0;
    for (int w = 0; w < b->W; ++w)
        if (!walkers || walkers[w]) total += b->hw[w].n;
    std::unique_ptr<int[]> acts(new int[total]);  // the free-atom lists (global ids), walker after walker
    for (int w = 0; w < b->W; ++w) {
        if (walkers && !walkers[w]) continue;
        const int off = b->hw[w].off, n = b->hw[w].n;
        const int *fr = frozen ? frozen + off : b->hfrozen.data() + off;
        int *act = acts.get() + iwords, m = 0;
        for (int i = 0; i < n; ++i)
            if (!fr[i]) act[m++] = off + i;
        LoadItem it{};
        it.walker = w;
        it.has_x = x0 ? 1 : 0;
        it.nact = m;
        it.dbl = (long long)dwords;
        it.ints = (long long)iwords;
        dwords += 3 * (size_t)m + (x0 ? 3 * (size_t)n : 0);
        iwords += m;
        items.push_back(it);
    }
    if (items.empty()) return AKMC_SUCCESS;
    const size_t ibytes = items.size() * sizeof(LoadItem);
    const size_t dbytes = dwords * sizeof(double), nbytes = iwords * sizeof(int);
    TRY(ensure_stage(b, ibytes + dbytes + nbytes + 64));
    char *base = (char *)b->stage_pin;
    double *D = (double *)(base + ibytes);
    int *I = (int *)(base + ibytes + dbytes);
    for (const LoadItem &it : items) {
        const int w = it.walker, off = b->hw[w].off, n = b->hw[w].n, m = it.nact;
        const int *act = acts.get() + it.ints;
        double *nw = D + it.dbl;
        double nn = 0.0;
        for (int c = 0; c < 3; ++c)
            for (int k = 0; k < m; ++k) {
                const double v = mode[c * A + act[k]];
                nw[(size_t)c * m + k] = v;
                nn += v * v;
            }
        if (nn <= 0.0) return fail(AKMC_EINVAL, "walker %d: zero start mode", w);
        nn = 1.0 / std::sqrt(nn);
        for (size_t k = 0; k < 3 * (size_t)m; ++k) nw[k] *= nn;
        if (x0)
            for (int c = 0; c < 3; ++c)
                std::memcpy(nw + 3 * (size_t)m + (size_t)c * n, x0 + c * A + off, n * sizeof(double));
        std::memcpy(I + it.ints, act, m * sizeof(int));
    }
    // every walker's data are good: the host's masks and lists become those
    // the device gets
    for (const LoadItem &it : items) {
        const int off = b->hw[it.walker].off, n = b->hw[it.walker].n;
        if (frozen) std::copy(frozen + off, frozen + off + n, b->hfrozen.begin() + off);
        std::copy(acts.get() + it.ints, acts.get() + it.ints + it.nact, b->hact.begin() + off);
        b->hnact[it.walker] = it.nact;
    }
    std::memcpy(base, items.data(), ibytes);
    HIPCHK(hipMemcpyAsync(b->stage_dev, b->stage_pin, ibytes + dbytes + nbytes, hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipEventRecord(b->stage_ev, b->stream));
    b->stage_pending = true;
    char *dbase = (char *)b->stage_dev;
    akmc_launch_load_walkers(b->d, b->s, (const LoadItem *)dbase, (int)items.size(), (const double *)(dbase + ibytes),
                             (const int *)(dbase + ibytes + dbytes), b->stream);
    HIPCHK(hipGetLastError());
    // queued behind a chunk in flight, the load returns at once
    if (!b->inflight) HIPCHK(hipStreamSynchronize(b->stream));
    return AKMC_SUCCESS;
}

int copy_walkers_out(akmc_batch_t b, const double *src, int nw, const int *walkers, double *out);
int copy_walkers_out3(akmc_batch_t b, const double *const src[3], int nw, const int *walkers, double *out);

int capture_graph(akmc_batch_t b, int steps, const ChunkPlan &plan)
{
    drop_graph(b);
    HIPCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    enqueue_steps(b, steps, plan);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(b->stream, &g);
    if (e != hipSuccess) return fail(AKMC_EHIP, "graph capture failed: %s", hipGetErrorString(e));
    b->graph = g;
    HIPCHK(hipGraphInstantiate(&b->gexec, g, nullptr, nullptr, 0));
    b->graph_steps = steps;
    b->graph_res = 2 * plan.res + plan.service;
    b->graph_args = b->s;
    b->graph_d = step_dev(b);
    b->graph_prec = batch_mode(b);
    return AKMC_SUCCESS;
}

}  // namespace

// ======================================================================
extern "C" {

const char *akmc_last_error(void) { return g_err.c_str(); }

int akmc_fail(int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

int akmc_version(void) { return 1; }

int akmc_field_create(const char *text, akmc_field_t *out)
{
    if (!out) return fail(AKMC_EINVAL, "null output handle");
    akmc_field_t f = new akmc_field_s();
    int rc = parse_potentials(f, text);
    if (rc != AKMC_SUCCESS) {
        delete f;
        return rc;
    }
    build_tables(f);
    *out = f;
    return AKMC_SUCCESS;
}

void akmc_field_destroy(akmc_field_t f)
{
    if (!f) return;
    if (f->single) batch_free(f->single);
    if (f->dev) (void)hipFree(f->dev);
    if (f->eam_dev) (void)hipFree(f->eam_dev);
    if (f->dsf_dev) (void)hipFree(f->dsf_dev);
    delete f;
}

int akmc_field_kind(akmc_field_t f) { return f ? f->kind : AKMC_EINVAL; }

int akmc_field_set_ewald(akmc_field_t f, double eta, int gx, int gy, int gz)
{
    if (!f || eta <= 0 || gx < 1 || gy < 1 || gz < 1) return fail(AKMC_EINVAL, "bad Ewald parameters");
    f->explicit_ewald = true;
    f->eta = eta;
    f->gcell[0] = gx;
    f->gcell[1] = gy;
    f->gcell[2] = gz;
    return AKMC_SUCCESS;
}

int akmc_field_set_skin(akmc_field_t f, double skin)
{
    if (!f || skin < 0) return fail(AKMC_EINVAL, "bad skin");
    f->skin = skin;
    build_tables(f);
    return AKMC_SUCCESS;
}

int akmc_field_set_list_density(akmc_field_t f, double atoms_per_A3)
{
    if (!f || !(atoms_per_A3 >= 0.0) || atoms_per_A3 > 10.0) return fail(AKMC_EINVAL, "bad list density");
    f->list_density = atoms_per_A3;
    return AKMC_SUCCESS;
}

int akmc_field_set_precision(akmc_field_t f, int bits)
{
    if (!f || (bits != 32 && bits != 64)) return fail(AKMC_EINVAL, "precision must be 32 or 64");
    f->fp64 = bits == 64;
    return AKMC_SUCCESS;
}

int akmc_field_setup(akmc_field_t f, const double lat[9], int max_atoms)
{
    if (!f || !lat || max_atoms <= 0) return fail(AKMC_EINVAL, "bad setup arguments");
    TRY(check_cell(f, lat));
    return ensure_single(f, max_atoms, lat);
}

int akmc_field_num_kvectors(akmc_field_t f) { return f ? f->nk_last : 0; }

}  // extern "C"

int akmc_field_view(akmc_field_s *f, FieldView *v)
{
    if (!f || !v) return fail(AKMC_EINVAL, "bad arguments");
    v->dev = f->dev;
    v->host = &f->host;
    v->rc = f->rc;
    v->skin = f->skin;
    v->kind = f->kind;
    v->min_image = f->min_image ? 1 : 0;
    v->eam = f->eam.empty() ? 0 : 1;
    v->fp64 = f->fp64;
    return AKMC_SUCCESS;
}

extern "C" {

int akmc_field_forces(akmc_field_t f, double *x, double *y, double *z, double *fx, double *fy, double *fz,
                      double stress[6], const double lat[9], const double *charge, const int *type,
                      const int *frozen, int n, akmc_energy *e)
{
    (void)frozen;  // unused by the reference's force call as well
    if (!f || !x || !y || !z || !fx || !fy || !fz || !type || n <= 0) return fail(AKMC_EINVAL, "bad arguments");
    if (f->kind == 1 && f->do_ewald && !charge) return fail(AKMC_EINVAL, "ionic field needs charges");
    TRY(ensure_single(f, n, lat));
    akmc_batch_t b = f->single;
    TRY(upload(b, x, y, z, type, charge, false));
    TRY(run_forces(b, stress != nullptr));
    if (pinned_io(b)) {
        TRY(fetch_all(b));
        const double *pf = (const double *)(b->io_pin + b->io_out);
        std::memcpy(fx, pf, n * sizeof(double));
        std::memcpy(fy, pf + n, n * sizeof(double));
        std::memcpy(fz, pf + 2 * (size_t)n, n * sizeof(double));
    } else {
        TRY(check_overflow(b));
        HIPCHK(hipMemcpyAsync(fx, b->d.fx, n * sizeof(double), hipMemcpyDeviceToHost, b->stream));
        HIPCHK(hipMemcpyAsync(fy, b->d.fy, n * sizeof(double), hipMemcpyDeviceToHost, b->stream));
        HIPCHK(hipMemcpyAsync(fz, b->d.fz, n * sizeof(double), hipMemcpyDeviceToHost, b->stream));
        TRY(fetch_out(b));
    }
    if (e) to_energy(b->hout[0], e);
    if (stress)
        for (int c = 0; c < 6; ++c) stress[c] = b->hout[0].stress[c];
    host_wrap(f->min_image, lat, n, x, y, z);
    return AKMC_SUCCESS;
}

int akmc_field_energy(akmc_field_t f, double *x, double *y, double *z, const double lat[9], const double *charge,
                      const int *type, int n, akmc_energy *e)
{
    if (!f || !x || !y || !z || !type || n <= 0) return fail(AKMC_EINVAL, "bad arguments");
    if (f->kind == 1 && f->do_ewald && !charge) return fail(AKMC_EINVAL, "ionic field needs charges");
    TRY(ensure_single(f, n, lat));
    akmc_batch_t b = f->single;
    TRY(upload(b, x, y, z, type, charge, false));
    // this launch's own copy of the batch descriptor carries the energy-only
    // flag: no force pass, and the energy-only short-range forms of the
    // two-body table (TwoBody.h:81-150: Morse adds C12/r^12).  Tabulated EAM
    // keeps its force pass (its pair energy comes from it).
    BatchDev d = b->d;
    d.energy_only = 1;
    akmc_launch_forces_impl(d, f->host, batch_mode(b), 0, b->stream);
    HIPCHK(hipGetLastError());
    if (pinned_io(b)) {
        TRY(fetch_all(b));
    } else {
        TRY(check_overflow(b));
        TRY(fetch_out(b));
    }
    if (e) to_energy(b->hout[0], e);
    host_wrap(f->min_image, lat, n, x, y, z);
    // the energy path of a tabulated EAM field doubles the pair term
    // (calculateManyBodyPairEnergy, potentials/metal/ManyBody.cpp:444-450)
    if (e && f->kind == 0 && !f->eam.empty()) {
        e->vdw *= 2.0;
        e->total = e->many + e->vdw;
    }
    return AKMC_SUCCESS;
}

int akmc_batch_create(akmc_field_t f, int nwalkers, const int *natoms, const double *lat, akmc_batch_t *out)
{
    if (!f || nwalkers <= 0 || !natoms || !lat || !out) return fail(AKMC_EINVAL, "bad batch arguments");
    akmc_batch_t b = new akmc_batch_s();
    int rc = batch_build(f, nwalkers, natoms, lat, b);
    if (rc != AKMC_SUCCESS) {
        batch_free(b);
        return rc;
    }
    *out = b;
    return AKMC_SUCCESS;
}

void akmc_batch_destroy(akmc_batch_t b) { batch_free(b); }

int akmc_batch_upload(akmc_batch_t b, const double *x, const double *y, const double *z, const int *type,
                      const double *charge, const int *frozen)
{
    (void)frozen;
    if (!b || !x || !y || !z || !type) return fail(AKMC_EINVAL, "bad arguments");
    return upload(b, x, y, z, type, charge);
}

int akmc_batch_download(akmc_batch_t b, double *x, double *y, double *z, double *fx, double *fy, double *fz)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    size_t A = b->A;
    if (x) HIPCHK(hipMemcpyAsync(x, b->d.x, A * sizeof(double), hipMemcpyDeviceToHost, b->stream));
    if (y) HIPCHK(hipMemcpyAsync(y, b->d.y, A * sizeof(double), hipMemcpyDeviceToHost, b->stream));
    if (z) HIPCHK(hipMemcpyAsync(z, b->d.z, A * sizeof(double), hipMemcpyDeviceToHost, b->stream));
    if (fx) HIPCHK(hipMemcpyAsync(fx, b->d.fx, A * sizeof(double), hipMemcpyDeviceToHost, b->stream));
    if (fy) HIPCHK(hipMemcpyAsync(fy, b->d.fy, A * sizeof(double), hipMemcpyDeviceToHost, b->stream));
    if (fz) HIPCHK(hipMemcpyAsync(fz, b->d.fz, A * sizeof(double), hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return AKMC_SUCCESS;
}

int akmc_batch_forces(akmc_batch_t b, akmc_energy *energies)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    TRY(run_forces(b, 0));
    TRY(check_overflow(b));
    TRY(fetch_out(b));
    if (energies)
        for (int w = 0; w < b->W; ++w) to_energy(b->hout[w], energies + w);
    return AKMC_SUCCESS;
}

int akmc_batch_forces_repeat(akmc_batch_t b, int nrep, double *ms)
{
    if (!b || nrep <= 0) return fail(AKMC_EINVAL, "bad arguments");
    HIPCHK(hipEventRecord(b->ev0, b->stream));
    for (int r = 0; r < nrep; ++r) TRY(run_forces(b, 0));
    HIPCHK(hipEventRecord(b->ev1, b->stream));
    HIPCHK(hipEventSynchronize(b->ev1));
    float t = 0.0f;
    HIPCHK(hipEventElapsedTime(&t, b->ev0, b->ev1));
    if (ms) *ms = t;
    return check_overflow(b);
}

int akmc_batch_set_variant(akmc_batch_t b, int lanes, int unroll)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    if (lanes != 1 && lanes != 2 && lanes != 4 && lanes != 8)
        return fail(AKMC_EINVAL, "lanes per atom must be 1, 2, 4 or 8, got %d", lanes);
    if (unroll != 1 && unroll != 2 && unroll != 4 && unroll != 8)
        return fail(AKMC_EINVAL, "unroll must be 1, 2, 4 or 8, got %d", unroll);
    if (b->d.lpa != lanes || b->d.unroll != unroll) drop_graph(b);  // the captured graph holds the old kernels
    b->d.lpa = lanes;
    b->d.unroll = unroll;
    return AKMC_SUCCESS;
}

int akmc_batch_set_staging(akmc_batch_t b, int on)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    if (on && !b->stage_ok)
        return fail(AKMC_EUNSUPPORTED,
                    "LDS staging needs a many-body field whose largest walker's gather records "
                    "(%d bytes) fit one workgroup's LDS", b->d.stage_bytes);
    if (b->d.staged != (on ? 1 : 0)) drop_graph(b);
    b->d.staged = on ? 1 : 0;
    return AKMC_SUCCESS;
}

int akmc_batch_staging(akmc_batch_t b, int *on, int *possible)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    if (on) *on = b->d.staged;
    if (possible) *possible = b->stage_ok ? 1 : 0;
    return AKMC_SUCCESS;
}

int akmc_batch_autotune(akmc_batch_t b, int nrep, int best[3], double ms[AKMC_NVARIANTS])
{
    if (!b || nrep <= 0) return fail(AKMC_EINVAL, "bad arguments");
    static const int lanes[4] = {1, 2, 4, 8}, unroll[4] = {1, 2, 4, 8};
    double t[AKMC_NVARIANTS];
    TRY(run_forces(b, 0));  // lists current before timing
    const int nv = b->stage_ok ? AKMC_NVARIANTS : AKMC_NVARIANTS / 2;
    for (int v = 0; v < AKMC_NVARIANTS; ++v) {
        t[v] = -1.0;
        if (v >= nv) continue;
        TRY(akmc_batch_set_staging(b, v / 16));
        TRY(akmc_batch_set_variant(b, lanes[v / 4 % 4], unroll[v % 4]));
        TRY(run_forces(b, 0));  // first launch of this instantiation
        TRY(akmc_batch_forces_repeat(b, nrep, &t[v]));
    }
    if (ms)
        for (int v = 0; v < AKMC_NVARIANTS; ++v) ms[v] = t[v];
    int k = 0;
    for (int v = 1; v < nv; ++v)
        if (t[v] < t[k]) k = v;
    TRY(akmc_batch_set_staging(b, k / 16));
    TRY(akmc_batch_set_variant(b, lanes[k / 4 % 4], unroll[k % 4]));
    if (best) {
        best[0] = lanes[k / 4 % 4];
        best[1] = unroll[k % 4];
        best[2] = k / 16;
    }
    return AKMC_SUCCESS;
}

int akmc_batch_total_atoms(akmc_batch_t b) { return b ? b->A : 0; }

long long akmc_batch_rebuilds(akmc_batch_t b)
{
    if (!b) return 0;
    unsigned long long v = 0;
    if (hipMemcpy(&v, akmc_rebuild_counter_ptr(), sizeof v, hipMemcpyDeviceToHost) != hipSuccess) return -1;
    return (long long)(v - b->rebuild_base);
}


void akmc_relax_defaults(akmc_relax_params *p)
{
    if (!p) return;
    p->maxIter = 3000;
    p->normTol = 1.0e-5;
    p->forceTol = 1.0e-4;
    p->N_min = 5;
    p->initTimeStep = 0.0005;
    p->alphaDecrease = 0.99;
    p->stepIncrease = 1.1;
    p->stepDecrease = 0.5;
    p->alphaStart = 0.1;
    p->maxTimeStep = 0.00075;
    p->timeStepUnit = 9648.530821;
    p->method = AKMC_RELAX_FIRE;
    p->verletIntegration = 0;
    p->N_delaySteps = 20;
    p->N_maxUphill = 50;
    p->initialDelay = 1;
    p->minTimeStep = 0.0001;
}

void akmc_dimer_defaults(akmc_dimer_params *p)
{
    if (!p) return;
    p->deltaTheta = 0.005;
    p->dimerDisplacement = 0.01;
    p->maxDeltaX = 0.5;
    p->maxRotations = 20;
    p->maxParIter = 1000;
    p->maxEigenvalue = 0.0;
    p->normTol = 0.1;
    p->forceTol = 1.0e-2;
    p->N_min = 5;
    p->alphaDecrease = 0.99;
    p->stepIncrease = 1.1;
    p->stepDecrease = 0.5;
    p->alphaStart = 0.1;
    p->initTimeStep = 0.005;
    p->maxTimeStep = 0.01;
    p->maxStep = 0.1;
    p->timeStepUnit = 9648.530821;
}

void akmc_art_defaults(akmc_art_params *p)
{
    if (!p) return;
    p->numLanczosVectors = 20;
    p->deltaX = 0.01;
    p->maxEigenvalue = 0.0;
    p->eigValTol = 0.001;
    p->parDamp = 0.5;
    p->maxParIter = 1000;
    p->normTol = 1.0e-4;
    p->forceTol = 1.0e-3;
    p->N_min = 5;
    p->initTimeStep = 0.005;
    p->alphaDecrease = 0.99;
    p->stepIncrease = 1.1;
    p->stepDecrease = 0.5;
    p->alphaStart = 0.1;
    p->maxTimeStep = 0.01;
    p->timeStepUnit = 9648.530821;
}

int akmc_batch_set_frozen(akmc_batch_t b, const int *frozen)
{
    if (!b || !frozen) return fail(AKMC_EINVAL, "bad arguments");
    TRY(search_alloc(b));
    HIPCHK(hipMemcpyAsync((void *)b->s.frozen, frozen, b->A * sizeof(int), hipMemcpyHostToDevice, b->stream));
    // a search under way whose free atoms change starts over with its zone,
    // and on the chain: the resident kernel's lists and fixed parts are those
    // of its old free atoms, and its buffers hold AKMC_RES_FREE of them
    const int fresh = AKMC_ZONE_FRESH, one = 1;
    std::vector<int> changed;
    for (int w = 0; w < b->W; ++w) {
        const int off = b->hw[w].off, n = b->hw[w].n;
        if (!(b->hzflag[w] & AKMC_ZONE_ON) || std::equal(frozen + off, frozen + off + n, b->hfrozen.begin() + off))
            continue;
        changed.push_back(w);
        HIPCHK(hipMemcpyAsync(b->zflag + w, &fresh, sizeof(int), hipMemcpyHostToDevice, b->stream));
        HIPCHK(hipMemcpyAsync(b->d.rebuild + w, &one, sizeof(int), hipMemcpyHostToDevice, b->stream));
    }
    std::copy(frozen, frozen + b->A, b->hfrozen.begin());
    TRY(upload_active(b, nullptr));  // (waits for the stream)
    for (int w : changed) b->hzflag[w] = b->zf_pin[w] = fresh;
    return AKMC_SUCCESS;
}

static int check_relax_method(const akmc_relax_params *p)
{
    if (p->method != AKMC_RELAX_FIRE && p->method != AKMC_RELAX_FIRE2 && p->method != AKMC_RELAX_NONE)
        return fail(AKMC_EINVAL, "relax method %d is not one of AKMC_RELAX_FIRE, _FIRE2, _NONE", p->method);
    return AKMC_SUCCESS;
}

int akmc_batch_start_relax(akmc_batch_t b, const int *walkers, const akmc_relax_params *p)
{
    if (!b || !p) return fail(AKMC_EINVAL, "bad arguments");
    TRY(search_alloc(b));
    TRY(check_relax_method(p));
    RelaxParamsDev &r = b->s.rp;
    r.normTol = p->normTol;
    r.forceTol = p->forceTol;
    r.initTimeStep = p->initTimeStep;
    r.maxTimeStep = p->maxTimeStep;
    r.alphaStart = p->alphaStart;
    r.alphaDecrease = p->alphaDecrease;
    r.stepIncrease = p->stepIncrease;
    r.stepDecrease = p->stepDecrease;
    r.timeStepUnit = p->timeStepUnit;
    r.minTimeStep = p->minTimeStep;
    r.maxIter = p->maxIter;
    r.N_min = p->N_min;
    r.method = p->method;
    r.verlet = p->verletIntegration ? 1 : 0;
    r.N_delaySteps = p->N_delaySteps;
    r.N_maxUphill = p->N_maxUphill;
    r.initialDelay = p->initialDelay ? 1 : 0;
    // velocities start at zero
    TRY(for_runs(b, walkers, [&](size_t off, size_t n) {
        for (int c = 0; c < 3; ++c)
            HIPCHK(hipMemsetAsync(b->s.V + (size_t)c * b->A + off, 0, n * sizeof(double), b->stream));
        return (int)AKMC_SUCCESS;
    }));
    return start_walkers(b, walkers, WK_RELAX, p->initTimeStep, p->alphaStart);
}

int akmc_batch_start_dimer(akmc_batch_t b, const int *walkers, const double *x0, const double *mode,
                           const int *frozen, const akmc_dimer_params *p)
{
    if (!b || !p || !mode) return fail(AKMC_EINVAL, "bad arguments");
    TRY(search_alloc(b));
    DimerParamsDev &d = b->s.dp;
    d.deltaTheta = p->deltaTheta;
    d.dimerDisplacement = p->dimerDisplacement;
    d.maxEigenvalue = p->maxEigenvalue;
    d.normTol = p->normTol;
    d.forceTol = p->forceTol;
    d.alphaStart = p->alphaStart;
    d.alphaDecrease = p->alphaDecrease;
    d.stepIncrease = p->stepIncrease;
    d.stepDecrease = p->stepDecrease;
    d.initTimeStep = p->initTimeStep;
    d.maxTimeStep = p->maxTimeStep;
    d.maxStep = p->maxStep;
    d.timeStepUnit = p->timeStepUnit;
    d.maxRotations = p->maxRotations;
    d.maxParIter = p->maxParIter;
    d.N_min = p->N_min;
    TRY(load_walkers(b, walkers, x0, mode, frozen));
    return start_walkers(b, walkers, WK_DIMER, p->initTimeStep, p->alphaStart);
}

int akmc_batch_start_art(akmc_batch_t b, const int *walkers, const double *x0, const double *mode,
                         const int *frozen, const akmc_art_params *p)
{
    if (!b || !p || !mode) return fail(AKMC_EINVAL, "bad arguments");
    if (p->numLanczosVectors < 2 || p->numLanczosVectors > AKMC_LZ_MAX)
        return fail(AKMC_EINVAL, "numLanczosVectors must be in [2, %d]", AKMC_LZ_MAX);
    TRY(search_alloc(b));
    TRY(ensure_lanczos(b));
    ARTParamsDev &a = b->s.ap;
    a.deltaX = p->deltaX;
    a.maxEigenvalue = p->maxEigenvalue;
    a.eigValTol = p->eigValTol;
    a.parDamp = p->parDamp;
    a.normTol = p->normTol;
    a.forceTol = p->forceTol;
    a.initTimeStep = p->initTimeStep;
    a.alphaDecrease = p->alphaDecrease;
    a.stepIncrease = p->stepIncrease;
    a.stepDecrease = p->stepDecrease;
    a.alphaStart = p->alphaStart;
    a.maxTimeStep = p->maxTimeStep;
    a.timeStepUnit = p->timeStepUnit;
    a.numLanczosVectors = p->numLanczosVectors;
    a.maxParIter = p->maxParIter;
    a.N_min = p->N_min;
    TRY(load_walkers(b, walkers, x0, mode, frozen));
    return start_walkers(b, walkers, WK_ART, p->initTimeStep, p->alphaStart);
}

}  // extern "C"

namespace {

// launches one chunk of `steps` micro-steps and the copies of the walker
// states and the overflow flag that its wait reads
int launch_chunk(akmc_batch_t b, int steps, int running)
{
    b->inflight_steps = 0;
    b->inflight = 1;
    if (running == 0) return AKMC_SUCCESS;
    // k micro-steps as one graph launch; the state kernels keep the
    // per-walker active flags current (0 when a walker ends, FP64 while
    // it verifies), so the host only reads states and the overflow flag
    if (b->ktimer && steps > akmc_batch_s::kTimerSteps) {
        b->inflight = 0;
        return fail(AKMC_EINVAL, "sync_every is limited to %d while the kernel timer runs", akmc_batch_s::kTimerSteps);
    }
    // HIP events recorded inside a replayed graph cannot be timed, so the
    // kernel timer launches the micro-steps one by one
    const ChunkPlan plan{resident_mode(b), parts_pending(b)};
    b->s.fire_on = 0;
    if (b->s.rp.method == AKMC_RELAX_FIRE && !b->s.rp.verlet)
        for (int w = 0; w < b->W && !b->s.fire_on; ++w)
            b->s.fire_on = b->hws[w].kind == WK_RELAX && b->hws[w].state != ST_DONE && b->hnact[w] == b->hw[w].n &&
                           b->hw[w].n <= AKMC_FIRE_ATOMS;
    TRY(sync_res_args(b));
    if (b->use_graphs && !b->ktimer) {
        const BatchDev bd = step_dev(b);
        if (!b->gexec || b->graph_steps != steps || b->graph_res != 2 * plan.res + plan.service || b->graph_prec != batch_mode(b) ||
            std::memcmp(&b->graph_args, &b->s, sizeof(SearchDev)) != 0 ||
            std::memcmp(&b->graph_d, &bd, sizeof(BatchDev)) != 0)
            TRY(capture_graph(b, steps, plan));
        HIPCHK(hipGraphLaunch(b->gexec, b->stream));
    } else {
        enqueue_steps(b, steps, plan);
        HIPCHK(hipGetLastError());
    }
    // the running resident walkers get their parts (the device clears the same
    // bits, and their current mode's)
    for (int w = 0; w < b->W; ++w)
        if ((b->hzflag[w] & AKMC_ZONE_RES) && b->hws[w].kind != WK_IDLE && b->hws[w].state != ST_DONE)
            b->hzflag[w] &= ~akmc_res_precisions(b->s);
    if (b->hv_on) {
        // the buffer the host read two waits ago
        b->hv_cur ^= 1;
        akmc_launch_harvest_pack(b->d, b->s, b->harvested, b->hv_dev[b->hv_cur], b->stream);
        HIPCHK(hipGetLastError());
        b->hv_inflight = b->hv_cur;
    }
    HIPCHK(hipMemcpyAsync(b->hws_pin, b->s.ws, b->W * sizeof(WalkerState), hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipMemcpyAsync(b->ov_pin, b->d.overflow, sizeof(int), hipMemcpyDeviceToHost, b->stream));
    b->inflight_steps = steps;
    return AKMC_SUCCESS;
}

}  // namespace

extern "C" {

int akmc_batch_run_async(akmc_batch_t b, int steps)
{
    if (!b || !b->search_alloc || steps < 1) return fail(AKMC_EINVAL, "bad arguments");
    if (b->inflight) return fail(AKMC_EINVAL, "a run chunk is already in flight");
    b->s.default_mode = batch_mode(b);  // the mode the state kernels give walkers they move on
    TRY(fetch_states(b));
    int running = 0;
    TRY(refresh_active(b, &running));
    return launch_chunk(b, steps, running);
}

int akmc_batch_run_next(akmc_batch_t b, int steps)
{
    if (!b || !b->search_alloc || steps < 1) return fail(AKMC_EINVAL, "bad arguments");
    if (b->inflight) return fail(AKMC_EINVAL, "a run chunk is already in flight");
    b->s.default_mode = batch_mode(b);
    // the host's copy of the states is the last wait's, with the starts
    // made since; the device keeps the active flags
    int running = 0;
    for (int w = 0; w < b->W; ++w) running += b->hws[w].kind != WK_IDLE && b->hws[w].state != ST_DONE;
    return launch_chunk(b, steps, running);
}

int akmc_batch_run_wait(akmc_batch_t b, int *steps_done, int *running)
{
    if (!b || !b->inflight) return fail(AKMC_EINVAL, "no run chunk in flight");
    b->inflight = 0;
    const int k = b->inflight_steps;
    int run = 0;
    if (k > 0) {
        HIPCHK(hipStreamSynchronize(b->stream));
        if (*b->ov_pin) return overflow_error(b, *b->ov_pin);
        if (b->ktimer && batch_mode(b) == 1 && b->f->host.kind == 0)
            for (int j = 0; j < k; ++j) {
                float t = 0.0f;
                HIPCHK(hipEventElapsedTime(&t, b->kev[0][j], b->kev[1][j]));
                b->kms += t;
                b->klaunches += 1;
            }
        std::memcpy(b->hws.data(), b->hws_pin, b->W * sizeof(WalkerState));
        for (int w = 0; w < b->W; ++w)  // its lists have outgrown the resident kernel
            if (b->hws[w].res & AKMC_RES_LEFT) b->hzflag[w] &= ~AKMC_ZONE_RES;
        if (b->hv_on) b->hv_last = b->hv_inflight;
    } else {
        HIPCHK(hipStreamSynchronize(b->stream));  // starts queued since the launch
    }
    // walkers started behind the chunk have not run yet
    for (const auto &p : b->started_inflight) {
        b->hws[p.first] = p.second;
        b->hzflag[p.first] = b->zf_pin[p.first];  // whether it fits the resident kernel
    }
    b->started_inflight.clear();
    for (int w = 0; w < b->W; ++w) run += b->hws[w].kind != WK_IDLE && b->hws[w].state != ST_DONE;
    if (steps_done) *steps_done = k;
    if (running) *running = run;
    return AKMC_SUCCESS;
}

int akmc_batch_set_harvest(akmc_batch_t b, int on)
{
    if (!b || !b->search_alloc) return fail(AKMC_EINVAL, "no search has been started");
    if (b->inflight) return fail(AKMC_EINVAL, "a run chunk is in flight");
    if (on && !b->harvested) {
        TRY(dalloc(b, &b->harvested, b->W));
        for (int k = 0; k < 2; ++k) {
            HIPCHK(hipHostMalloc((void **)&b->hv_pin[k], 3 * (size_t)b->A * sizeof(double), hipHostMallocDefault));
            HIPCHK(hipHostGetDevicePointer((void **)&b->hv_dev[k], b->hv_pin[k], 0));
        }
    }
    // walkers that have already ended are harvested by the next chunk
    if (on) HIPCHK(hipMemsetAsync(b->harvested, 0, b->W * sizeof(int), b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    b->hv_on = on ? 1 : 0;
    b->hv_last = -1;
    return AKMC_SUCCESS;
}

int akmc_batch_get_harvested_positions(akmc_batch_t b, int nw, const int *walkers, double *out)
{
    if (!b || nw < 0 || (nw && (!walkers || !out))) return fail(AKMC_EINVAL, "bad arguments");
    if (!b->hv_on || b->hv_last < 0) return fail(AKMC_EINVAL, "no harvested chunk has been waited for");
    const double *src = b->hv_pin[b->hv_last];
    const size_t A = b->A;
    size_t o = 0;
    for (int k = 0; k < nw; ++k) {
        const int w = walkers[k];
        if (w < 0 || w >= b->W) return fail(AKMC_EINVAL, "walker %d out of range", w);
        const int off = b->hw[w].off, n = b->hw[w].n;
        for (int c = 0; c < 3; ++c, o += n) std::memcpy(out + o, src + c * A + off, n * sizeof(double));
    }
    return AKMC_SUCCESS;
}

int akmc_batch_run(akmc_batch_t b, int max_steps, int sync_every, int *steps_done)
{
    if (!b || !b->search_alloc || max_steps < 0 || sync_every < 1) return fail(AKMC_EINVAL, "bad arguments");
    int done = 0, running = 1;
    while (running > 0 && done < max_steps) {
        int k = std::min(sync_every, max_steps - done), got = 0;
        // nothing but the chunks changes the walkers from here on
        TRY(done == 0 ? akmc_batch_run_async(b, k) : akmc_batch_run_next(b, k));
        TRY(akmc_batch_run_wait(b, &got, &running));
        if (got == 0) break;
        done += got;
    }
    if (steps_done) *steps_done = done;
    return AKMC_SUCCESS;
}

int akmc_batch_kernel_timer(akmc_batch_t b, int enable)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    if (enable)
        for (auto &row : b->kev)
            for (auto &e : row)
                if (!e) HIPCHK(hipEventCreate(&e));
    b->ktimer = enable != 0;
    b->kms = 0.0;
    b->klaunches = 0;
    return AKMC_SUCCESS;
}

int akmc_batch_eval_counts(akmc_batch_t b, long long *counts)
{
    if (!b || !counts) return fail(AKMC_EINVAL, "bad arguments");
    if (!b->search_alloc) {
        for (int w = 0; w < b->W; ++w) counts[w] = 0;
        return AKMC_SUCCESS;
    }
    HIPCHK(hipMemcpy(counts, b->s.evals32, b->W * sizeof(long long), hipMemcpyDeviceToHost));
    return AKMC_SUCCESS;
}

int akmc_batch_kernel_time(akmc_batch_t b, double *ms, long long *launches)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    if (ms) *ms = b->kms;
    if (launches) *launches = b->klaunches;
    return AKMC_SUCCESS;
}

int akmc_batch_set_graphs(akmc_batch_t b, int enable)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    b->use_graphs = enable != 0;
    if (!b->use_graphs) drop_graph(b);
    return AKMC_SUCCESS;
}

int akmc_batch_set_logic_block(akmc_batch_t b, int threads)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    if (threads != 256 && threads != 1024) return fail(AKMC_EINVAL, "threads must be 256 or 1024, got %d", threads);
    b->logic_wide = threads == 1024;
    drop_graph(b);
    return AKMC_SUCCESS;
}

int akmc_batch_set_search_zone(akmc_batch_t b, int enable)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    b->zone_on = enable != 0;
    drop_graph(b);
    return AKMC_SUCCESS;
}

int akmc_batch_set_resident(akmc_batch_t b, int enable)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    b->res_on = enable != 0;
    return AKMC_SUCCESS;
}

int akmc_batch_set_search_variant(akmc_batch_t b, const int v[9])
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    int nv[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    auto ok = [](int x) { return x == 1 || x == 2 || x == 4 || x == 8; };
    if (v) {
        for (int p = 0; p < 3; ++p) {
            const int l = v[3 * p], u = v[3 * p + 1], st = v[3 * p + 2];
            if (l == 0) continue;
            if (!ok(l) || !ok(u)) return fail(AKMC_EINVAL, "part %d: lanes and unroll must be 1, 2, 4 or 8", p + 1);
            if (st && !b->stage_ok) return fail(AKMC_EUNSUPPORTED, "LDS staging is not possible for this batch");
            nv[3 * p] = l;
            nv[3 * p + 1] = u;
            nv[3 * p + 2] = st ? 1 : 0;
        }
    }
    std::memcpy(b->sv, nv, sizeof nv);
    drop_graph(b);
    return AKMC_SUCCESS;
}

static int time_search_phases_prec(akmc_batch_t b, int prec, int nrep, bool chain, double ms[4]);

// The variants are those of the chain's pair kernels.  What they do for a
// resident walker is the evaluation of all its atoms on its first micro-step,
// so that is what they are timed on: the flags that ask for it are set while
// the object lives.
struct FullEvaluations {
    akmc_batch_t b;
    std::vector<int> flags;
    explicit FullEvaluations(akmc_batch_t b_) : b(b_) {}
    int set()
    {
        flags.resize(b->W);
        HIPCHK(hipMemcpyAsync(flags.data(), b->zflag, b->W * sizeof(int), hipMemcpyDeviceToHost, b->stream));
        HIPCHK(hipStreamSynchronize(b->stream));
        std::vector<int> full = flags;
        for (int &f : full)
            if (f & AKMC_ZONE_RES) f |= AKMC_ZONE_FULL32 | AKMC_ZONE_FULL64;
        HIPCHK(hipMemcpyAsync(b->zflag, full.data(), b->W * sizeof(int), hipMemcpyHostToDevice, b->stream));
        HIPCHK(hipStreamSynchronize(b->stream));
        return AKMC_SUCCESS;
    }
    // resident walkers' flags as they were (the chain keeps the others')
    ~FullEvaluations()
    {
        std::vector<int> now(flags.size());
        const size_t n = now.size() * sizeof(int);
        if (!n || hipMemcpy(now.data(), b->zflag, n, hipMemcpyDeviceToHost) != hipSuccess) return;
        for (size_t w = 0; w < now.size(); ++w)
            if (now[w] & AKMC_ZONE_RES) now[w] = flags[w];
        (void)hipMemcpy(b->zflag, now.data(), n, hipMemcpyHostToDevice);
    }
};

int akmc_batch_autotune_search(akmc_batch_t b, int nrep, int best[9], double ms1[AKMC_NVARIANTS],
                               double ms2[AKMC_NVARIANTS], double ms64[AKMC_NVARIANTS])
{
    if (!b || nrep <= 0) return fail(AKMC_EINVAL, "bad arguments");
    if (!b->search_alloc) return fail(AKMC_EINVAL, "no search has been started");
    static const int lanes[4] = {1, 2, 4, 8}, unroll[4] = {1, 2, 4, 8};
    const int nv = b->stage_ok ? AKMC_NVARIANTS : AKMC_NVARIANTS / 2;
    double t1[AKMC_NVARIANTS], t2[AKMC_NVARIANTS], ms[4];
    FullEvaluations full(b);
    TRY(full.set());
    for (int v = 0; v < AKMC_NVARIANTS; ++v) {
        t1[v] = t2[v] = -1.0;
        if (v >= nv) continue;
        const int sv[9] = {lanes[v / 4 % 4], unroll[v % 4], v / 16, lanes[v / 4 % 4], unroll[v % 4], v / 16, 0, 0, 0};
        TRY(akmc_batch_set_search_variant(b, sv));
        TRY(time_search_phases_prec(b, batch_mode(b), 1, true, ms));  // first launch of this instantiation
        TRY(time_search_phases_prec(b, batch_mode(b), nrep, true, ms));
        t1[v] = ms[1];
        t2[v] = ms[2];
    }
    int k1 = 0, k2 = 0;
    for (int v = 1; v < nv; ++v) {
        if (t1[v] < t1[k1]) k1 = v;
        if (t2[v] < t2[k2]) k2 = v;
    }
    // the FP64 passes of mixed steps, on the walkers under FP64 verification
    // at the moment: both passes together
    double t64[AKMC_NVARIANTS];
    int k64 = 0;
    for (int v = 0; v < AKMC_NVARIANTS; ++v) {
        t64[v] = -1.0;
        if (v >= nv) continue;
        const int sv[9] = {0, 0, 0, 0, 0, 0, lanes[v / 4 % 4], unroll[v % 4], v / 16};
        TRY(akmc_batch_set_search_variant(b, sv));
        TRY(time_search_phases_prec(b, 2 | 4, 1, true, ms));
        TRY(time_search_phases_prec(b, 2 | 4, nrep, true, ms));
        t64[v] = ms[1] + ms[2];
        if (t64[v] < t64[k64]) k64 = v;
    }
    const int sv[9] = {lanes[k1 / 4 % 4], unroll[k1 % 4], k1 / 16, lanes[k2 / 4 % 4], unroll[k2 % 4], k2 / 16,
                       lanes[k64 / 4 % 4], unroll[k64 % 4], k64 / 16};
    TRY(akmc_batch_set_search_variant(b, sv));
    if (best) std::memcpy(best, sv, sizeof sv);
    for (int v = 0; v < AKMC_NVARIANTS; ++v) {
        if (ms1) ms1[v] = t1[v];
        if (ms2) ms2[v] = t2[v];
        if (ms64) ms64[v] = t64[v];
    }
    return AKMC_SUCCESS;
}

int akmc_batch_status(akmc_batch_t b, akmc_walker_status *out)
{
    if (!b || !out) return fail(AKMC_EINVAL, "bad arguments");
    if (!b->search_alloc) return fail(AKMC_EINVAL, "no search has been started");
    // while a run chunk is in flight: the states at the end of the previous
    // chunk, with the starts made since
    if (!b->inflight) TRY(fetch_states(b));
    for (int w = 0; w < b->W; ++w) {
        const WalkerState &ws = b->hws[w];
        out[w].kind = ws.kind;
        out[w].status = ws.status;
        out[w].done = ws.state == ST_DONE ? 1 : 0;
        out[w].iterations = ws.it;
        out[w].force_calls = ws.fcalls;
        out[w].energy = ws.E0;
        out[w].curvature = ws.C;
        out[w].verified = ws.verified_state;
        out[w].energy32 = ws.e32;
        out[w].curvature32 = ws.c32;
        out[w].energy64 = ws.e64;
        out[w].fmax64 = ws.fmax64;
        out[w].lambda1 = ws.lam1;
        out[w].lambda2 = ws.lam2;
        out[w].new_basin = ws.b2_new;
        out[w].basin2_status = ws.b2_status;
        out[w].basin2_force_calls = ws.b2_calls;
        out[w].basin2_iterations = ws.b2_iters;
        out[w].energy_basin2 = ws.eb2;
        out[w].energy_basin2_64 = ws.eb2_64;
        out[w].basin2_max_disp = std::sqrt(ws.b2_maxd2);
    }
    return AKMC_SUCCESS;
}

int akmc_batch_get_positions(akmc_batch_t b, double *x, double *y, double *z)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    size_t A = b->A;
    // before the first search or relax the batch's own positions are current
    const double *src[3] = {b->d.x, b->d.y, b->d.z};
    if (b->search_alloc) {
        src[0] = b->s.X;
        src[1] = b->s.X + A;
        src[2] = b->s.X + 2 * A;
    }
    HIPCHK(hipStreamSynchronize(b->stream));
    if (x) HIPCHK(hipMemcpy(x, src[0], A * sizeof(double), hipMemcpyDeviceToHost));
    if (y) HIPCHK(hipMemcpy(y, src[1], A * sizeof(double), hipMemcpyDeviceToHost));
    if (z) HIPCHK(hipMemcpy(z, src[2], A * sizeof(double), hipMemcpyDeviceToHost));
    return AKMC_SUCCESS;
}

int akmc_batch_get_walkers_positions(akmc_batch_t b, int nw, const int *walkers, double *out)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    if (b->search_alloc) return copy_walkers_out(b, b->s.X, nw, walkers, out);
    const double *const src[3] = {b->d.x, b->d.y, b->d.z};
    return copy_walkers_out3(b, src, nw, walkers, out);
}

int akmc_batch_get_walkers_saddles(akmc_batch_t b, int nw, const int *walkers, double *out)
{
    if (!b || !b->search_alloc || !b->s.Xs) return fail(AKMC_EINVAL, "the basin-2 stage has not been set up");
    return copy_walkers_out(b, b->s.Xs, nw, walkers, out);
}

}  // extern "C"

namespace {

// the [3][n] slices of src ([3][A]) of the listed walkers, one pinned
// transfer
int copy_walkers_out(akmc_batch_t b, const double *src, int nw, const int *walkers, double *out)
{
    const double *const c3[3] = {src, src + b->A, src + 2 * (size_t)b->A};
    return copy_walkers_out3(b, c3, nw, walkers, out);
}

// the flagged walkers' (3, n_w) slices of three [A] component arrays, packed
// walker after walker, through the pinned staging buffer
int copy_walkers_out3(akmc_batch_t b, const double *const src[3], int nw, const int *walkers, double *out)
{
    if (nw < 0 || (nw && (!walkers || !out))) return fail(AKMC_EINVAL, "bad arguments");
    size_t total = 0;
    for (int k = 0; k < nw; ++k) {
        if (walkers[k] < 0 || walkers[k] >= b->W) return fail(AKMC_EINVAL, "walker %d out of range", walkers[k]);
        total += 3 * (size_t)b->hw[walkers[k]].n;
    }
    if (nw == 0) return AKMC_SUCCESS;
    // one buffer: walker ids, their output offsets, then the packed doubles
    const size_t ibytes = ((size_t)nw * sizeof(int) + 7) / 8 * 8, obytes = (size_t)nw * sizeof(long long);
    const size_t need = ibytes + obytes + total * sizeof(double);
    if (need > b->gat_n) {
        if (b->gat_pin) HIPCHK(hipHostFree(b->gat_pin));
        if (b->gat_dev) HIPCHK(hipFree(b->gat_dev));
        b->gat_pin = b->gat_dev = nullptr;
        b->gat_n = 0;
        const size_t cap = need + need / 2;
        HIPCHK(hipHostMalloc((void **)&b->gat_pin, cap, hipHostMallocDefault));
        HIPCHK(hipMalloc((void **)&b->gat_dev, cap));
        b->gat_n = cap;
    }
    // while a run chunk is in flight the copy runs beside it on a side
    // stream (the walkers that had ended before the chunk are not written)
    hipStream_t st = b->stream;
    if (b->inflight) {
        if (!b->side) HIPCHK(hipStreamCreateWithFlags(&b->side, hipStreamNonBlocking));
        st = b->side;
    }
    int *ws = reinterpret_cast<int *>(b->gat_pin);
    long long *dst = reinterpret_cast<long long *>(b->gat_pin + ibytes);
    long long o = 0;
    for (int k = 0; k < nw; ++k) {
        ws[k] = walkers[k];
        dst[k] = o;
        o += 3 * (long long)b->hw[walkers[k]].n;
    }
    HIPCHK(hipMemcpyAsync(b->gat_dev, b->gat_pin, ibytes + obytes, hipMemcpyHostToDevice, st));
    double *dout = reinterpret_cast<double *>(b->gat_dev + ibytes + obytes);
    akmc_launch_gather_walkers(b->d.walkers, src, reinterpret_cast<const int *>(b->gat_dev),
                               reinterpret_cast<const long long *>(b->gat_dev + ibytes), nw, dout, st);
    HIPCHK(hipGetLastError());
    double *hout = reinterpret_cast<double *>(b->gat_pin + ibytes + obytes);
    HIPCHK(hipMemcpyAsync(hout, dout, total * sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    std::memcpy(out, hout, total * sizeof(double));
    return AKMC_SUCCESS;
}

}  // namespace

extern "C" {

int akmc_batch_get_walker_positions(akmc_batch_t b, int walker, double *x, double *y, double *z)
{
    if (!b || walker < 0 || walker >= b->W) return fail(AKMC_EINVAL, "bad arguments");
    size_t A = b->A, off = b->hw[walker].off, n = b->hw[walker].n;
    double *dst[3] = {x, y, z};
    const double *src[3] = {b->d.x, b->d.y, b->d.z};  // before the first search or relax
    if (b->search_alloc)
        for (int c = 0; c < 3; ++c) src[c] = b->s.X + c * A;
    for (int c = 0; c < 3; ++c)
        if (dst[c]) HIPCHK(hipMemcpyAsync(dst[c], src[c] + off, n * sizeof(double), hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return AKMC_SUCCESS;
}

int akmc_batch_get_mode(akmc_batch_t b, double *mode)
{
    if (!b || !b->search_alloc || !mode) return fail(AKMC_EINVAL, "no search state");
    HIPCHK(hipMemcpy(mode, b->s.N, 3 * (size_t)b->A * sizeof(double), hipMemcpyDeviceToHost));
    return AKMC_SUCCESS;
}


int akmc_batch_time_phases(akmc_batch_t b, int nrep, double ms[4])
{
    if (!b || nrep <= 0 || !ms) return fail(AKMC_EINVAL, "bad arguments");
    for (auto &e : b->evp)
        if (!e) HIPCHK(hipEventCreate(&e));
    for (int ph = 0; ph < 4; ++ph) ms[ph] = 0.0;
    for (int r = 0; r < nrep; ++r) {
        HIPCHK(hipEventRecord(b->evp[0], b->stream));
        for (int ph = 0; ph < 4; ++ph) {
            akmc_launch_phase(b->d, b->f->host, batch_mode(b), 0, ph, b->stream);
            HIPCHK(hipEventRecord(b->evp[ph + 1], b->stream));
        }
        HIPCHK(hipEventSynchronize(b->evp[4]));
        for (int ph = 0; ph < 4; ++ph) {
            float t = 0.0f;
            HIPCHK(hipEventElapsedTime(&t, b->evp[ph], b->evp[ph + 1]));
            ms[ph] += t;
        }
    }
    return check_overflow(b);
}

int akmc_batch_time_search_phases(akmc_batch_t b, int nrep, double ms[4])
{
    if (!b || nrep <= 0 || !ms) return fail(AKMC_EINVAL, "bad arguments");
    if (!b->search_alloc) return fail(AKMC_EINVAL, "no search has been started");
    return time_search_phases_prec(b, batch_mode(b), nrep, false, ms);
}

// per-phase times of nrep evaluations of the search walkers of precision
// mask prec (2 | 4: the FP64 passes of mixed steps) at their probes; chain:
// by the pair kernels alone
static int time_search_phases_prec(akmc_batch_t b, int prec, int nrep, bool chain, double ms[4])
{
    for (auto &e : b->evp)
        if (!e) HIPCHK(hipEventCreate(&e));
    const BatchDev d = step_dev(b);
    const int res = chain ? 0 : resident_mode(b);
    TRY(sync_res_args(b));
    for (int ph = 0; ph < 4; ++ph) ms[ph] = 0.0;
    for (int r = 0; r < nrep; ++r) {
        HIPCHK(hipEventRecord(b->evp[0], b->stream));
        for (int ph = 0; ph < 4; ++ph) {
            akmc_launch_phase(d, b->f->host, prec, 0, ph, b->stream);
            // resident walkers: their whole evaluation is timed with pass 1
            if (ph == 1 && res) {
                akmc_launch_res_base(d, b->f->host, akmc_res_precisions(b->s), b->stream);
                akmc_launch_search_resident(b->W, b->f->host, b->res_args, 1, 0, 1, b->stream);
            }
            HIPCHK(hipEventRecord(b->evp[ph + 1], b->stream));
        }
        HIPCHK(hipEventSynchronize(b->evp[4]));
        for (int ph = 0; ph < 4; ++ph) {
            float t = 0.0f;
            HIPCHK(hipEventElapsedTime(&t, b->evp[ph], b->evp[ph + 1]));
            ms[ph] += t;
        }
    }
    return check_overflow(b);
}

int akmc_batch_get_zone(akmc_batch_t b, int *member, int *size, int *flags, int *active)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    if (!b->search_alloc) return fail(AKMC_EINVAL, "no search has been started");
    if (member) HIPCHK(hipMemcpyAsync(member, b->zmark, b->A * sizeof(int), hipMemcpyDeviceToHost, b->stream));
    if (size) HIPCHK(hipMemcpyAsync(size, b->nz, b->W * sizeof(int), hipMemcpyDeviceToHost, b->stream));
    if (flags) HIPCHK(hipMemcpyAsync(flags, b->zflag, b->W * sizeof(int), hipMemcpyDeviceToHost, b->stream));
    if (active) HIPCHK(hipMemcpyAsync(active, b->d.active, b->W * sizeof(int), hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return AKMC_SUCCESS;
}

int akmc_batch_save_basin(akmc_batch_t b) { return akmc_batch_set_basins(b, nullptr, nullptr); }

int akmc_batch_set_basins(akmc_batch_t b, const int *walkers, const double *x)
{
    if (!b) return fail(AKMC_EINVAL, "bad arguments");
    TRY(search_alloc(b));  // search positions start at the resident ones
    if (!b->basin) TRY(dalloc(b, &b->basin, 3 * (size_t)b->A));
    b->s.basin = b->basin;
    const size_t A = b->A;
    if (!walkers && !x) {
        HIPCHK(hipMemcpyAsync(b->basin, b->s.X, 3 * A * sizeof(double), hipMemcpyDeviceToDevice, b->stream));
    } else {
        for (int w = 0; w < b->W; ++w) {
            if (walkers && !walkers[w]) continue;
            for (int c = 0; c < 3; ++c) {
                const size_t o = c * A + b->hw[w].off;
                if (x)
                    HIPCHK(hipMemcpyAsync(b->basin + o, x + o, b->hw[w].n * sizeof(double), hipMemcpyHostToDevice,
                                          b->stream));
                else
                    HIPCHK(hipMemcpyAsync(b->basin + o, b->s.X + o, b->hw[w].n * sizeof(double),
                                          hipMemcpyDeviceToDevice, b->stream));
            }
        }
    }
    HIPCHK(hipStreamSynchronize(b->stream));
    return AKMC_SUCCESS;
}

void akmc_basin2_defaults(akmc_basin2_params *p)
{
    if (!p) return;
    p->basin2Delta = 0.2;
    p->kmcBasinRadius = 0.5;  // docs/examples/gdc/control:11
    p->kmcMaxRadius = 5.0;
}

int akmc_batch_set_basin2(akmc_batch_t b, const akmc_basin2_params *p)
{
    if (!b) return fail(AKMC_EINVAL, "null batch");
    TRY(search_alloc(b));
    if (!p) {
        b->s.basin2_on = 0;
        b->s.final64 = 0;
        return AKMC_SUCCESS;
    }
    if (!(p->basin2Delta >= 0.0) || !(p->kmcBasinRadius >= 0.0) || !(p->kmcMaxRadius >= 0.0))
        return fail(AKMC_EINVAL, "basin2Delta, kmcBasinRadius and kmcMaxRadius must be >= 0");
    if (!b->s.Xs) TRY(dalloc(b, &b->s.Xs, 3 * (size_t)b->A));
    b->s.basin2_delta = p->basin2Delta;
    b->s.basin_r2 = p->kmcBasinRadius * p->kmcBasinRadius;
    b->s.max_r2 = p->kmcMaxRadius * p->kmcMaxRadius;
    b->s.basin2_on = 1;
    b->s.final64 = 1;
    return AKMC_SUCCESS;
}

int akmc_batch_start_relax_at(akmc_batch_t b, const int *walkers, const double *x0, const int *frozen,
                              const akmc_relax_params *p)
{
    if (!b || !p) return fail(AKMC_EINVAL, "bad arguments");
    TRY(check_relax_method(p));  // before the masks of running walkers change
    TRY(search_alloc(b));
    const size_t A = b->A;
    TRY(for_runs(b, walkers, [&](size_t off, size_t n) {
        if (frozen) {
            std::copy(frozen + off, frozen + off + n, b->hfrozen.begin() + off);
            HIPCHK(hipMemcpyAsync((void *)(b->s.frozen + off), frozen + off, n * sizeof(int), hipMemcpyHostToDevice,
                                  b->stream));
        }
        if (x0)
            for (int c = 0; c < 3; ++c)
                HIPCHK(hipMemcpyAsync(b->s.X + c * A + off, x0 + c * A + off, n * sizeof(double),
                                      hipMemcpyHostToDevice, b->stream));
        return (int)AKMC_SUCCESS;
    }));
    HIPCHK(hipStreamSynchronize(b->stream));
    if (frozen) TRY(upload_active(b, walkers));
    return akmc_batch_start_relax(b, walkers, p);
}

int akmc_batch_cancel(akmc_batch_t b, const int *walkers)
{
    if (!b || !b->search_alloc) return fail(AKMC_EINVAL, "no search state");
    TRY(fetch_states(b));
    for (int w = 0; w < b->W; ++w)
        if (!walkers || walkers[w]) b->hws[w].kind = WK_IDLE;
    HIPCHK(hipMemcpyAsync(b->s.ws, b->hws.data(), b->W * sizeof(WalkerState), hipMemcpyHostToDevice, b->stream));
    int run;
    return refresh_active(b, &run);
}

int akmc_batch_restore_basin(akmc_batch_t b, const int *walkers)
{
    if (!b || !b->basin) return fail(AKMC_EINVAL, "no saved basin");
    size_t A = b->A;
    for (int w = 0; w < b->W; ++w) {
        if (walkers && !walkers[w]) continue;
        for (int c = 0; c < 3; ++c) {
            size_t o = c * A + b->hw[w].off;
            HIPCHK(hipMemcpyAsync(b->s.X + o, b->basin + o, b->hw[w].n * sizeof(double), hipMemcpyDeviceToDevice,
                                  b->stream));
        }
        if (!walkers) break;
    }
    if (!walkers)
        HIPCHK(hipMemcpyAsync(b->s.X, b->basin, 3 * A * sizeof(double), hipMemcpyDeviceToDevice, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return AKMC_SUCCESS;
}


int akmc_batch_set_verify(akmc_batch_t b, int nl, double delta)
{
    if (!b || nl < 0 || nl > AKMC_LZ_MAX || (nl > 0 && delta <= 0.0))
        return fail(AKMC_EINVAL, "verification needs 0 <= nl <= %d and delta > 0", AKMC_LZ_MAX);
    TRY(search_alloc(b));
    if (nl > 0) TRY(ensure_lanczos(b));
    if (nl > 0 && (size_t)nl > (size_t)AKMC_LZ_MAX) return fail(AKMC_EINVAL, "nl too large");
    b->s.verify_nl = nl;
    b->s.verify_delta = delta;
    drop_graph(b);
    return AKMC_SUCCESS;
}

int akmc_batch_search_energies(akmc_batch_t b, int bits, double *energies)
{
    if (!b || !b->search_alloc || !energies || (bits != 32 && bits != 64))
        return fail(AKMC_EINVAL, "bad arguments");
    size_t A = b->A;
    HIPCHK(hipMemcpyAsync(b->d.x, b->s.X, A * sizeof(double), hipMemcpyDeviceToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(b->d.y, b->s.X + A, A * sizeof(double), hipMemcpyDeviceToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(b->d.z, b->s.X + 2 * A, A * sizeof(double), hipMemcpyDeviceToDevice, b->stream));
    std::vector<int> mode(b->W, bits == 64 ? 2 : 1);
    HIPCHK(hipMemcpyAsync(b->d.active, mode.data(), b->W * sizeof(int), hipMemcpyHostToDevice, b->stream));
    akmc_launch_forces_impl(b->d, b->f->host, bits == 64 ? 2 : 1, 0, b->stream);
    HIPCHK(hipGetLastError());
    TRY(check_overflow(b));
    TRY(fetch_out(b));
    for (int w = 0; w < b->W; ++w) energies[w] = b->hout[w].total;
    return AKMC_SUCCESS;
}

}  // extern "C"

// ------------------------------------------------------------------ MLP

struct akmc_mlp_s {
    int rows = 0;
    unsigned seed = 0;
    hipStream_t stream = nullptr;
    std::vector<void *> allocs;
    float *p = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;
    uint16_t *w1t = nullptr, *w2t = nullptr, *w3t = nullptr, *w2r = nullptr, *w3r = nullptr;
    float *X = nullptr, *T = nullptr, *Y = nullptr, *P = nullptr, *ms = nullptr;  // ms: mean and scale of the inputs
    char *rbuf = nullptr;  // the gradient's per-row operands
    double *lpart = nullptr;
    int adam_t = 0;
};

namespace {
template <typename T>
int malloc_m(akmc_mlp_t m, T **p, size_t n)
{
    HIPCHK(hipMalloc((void **)p, (n ? n : 1) * sizeof(T)));
    m->allocs.push_back((void *)*p);
    return AKMC_SUCCESS;
}

void mlp_free(akmc_mlp_t m)
{
    if (!m) return;
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    for (void *q : m->allocs) (void)hipFree(q);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

int mlp_refresh_weights(akmc_mlp_t m)
{
    akmc_mlp_launch_weights(m->p, m->w1t, m->w2t, m->w3t, m->w2r, m->w3r, m->stream);
    HIPCHK(hipGetLastError());
    return AKMC_SUCCESS;
}

// the inputs' mean and scale on the device (null: none)
int mlp_scaling(akmc_mlp_t m, const float *mean, const float *scale)
{
    if (!mean) return AKMC_SUCCESS;
    HIPCHK(hipMemcpyAsync(m->ms, mean, 48 * sizeof(float), hipMemcpyHostToDevice, m->stream));
    HIPCHK(hipMemcpyAsync(m->ms + 48, scale, 48 * sizeof(float), hipMemcpyHostToDevice, m->stream));
    return AKMC_SUCCESS;
}

// gradient sums of rows idx of (X, T), then the gradient (and, with step, the
// Adam step); acc: where the rows' mean loss is added, or null
int mlp_grad(akmc_mlp_t m, const float *X, const float *T, const int *idx, int M, int step, float lr, double *acc)
{
    akmc_mlp_launch_grad(X, T, idx, M, m->p, m->w1t, m->w2t, m->w3t, m->w2r, m->w3r, m->rbuf, m->P,
                         m->lpart, m->g, m->stream);
    if (step) ++m->adam_t;
    akmc_mlp_launch_update(m->P, M, m->g, m->p, m->m1, m->m2, m->w1t, m->w2t, m->w3t, m->w2r, m->w3r, step, lr,
                           std::max(m->adam_t, 1), m->lpart, acc, m->stream);
    HIPCHK(hipGetLastError());
    return AKMC_SUCCESS;
}
}  // namespace

extern "C" {

int akmc_mlp_create(int max_rows, unsigned seed, akmc_mlp_t *out)
{
    if (max_rows <= 0 || !out) return fail(AKMC_EINVAL, "bad arguments");
    akmc_mlp_t m = new akmc_mlp_s();
    m->rows = (max_rows + 255) / 256 * 256;
    m->seed = seed;
    auto bad = [&](int rc) {
        mlp_free(m);
        return rc;
    };
    if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess)
        return bad(fail(AKMC_EHIP, "stream creation failed"));
    const size_t R = m->rows, NP = AKMC_MLP_NPARAM;
    int rc = AKMC_SUCCESS;
    if ((rc = malloc_m(m, &m->p, NP)) || (rc = malloc_m(m, &m->g, NP)) || (rc = malloc_m(m, &m->m1, NP)) ||
        (rc = malloc_m(m, &m->m2, NP)) || (rc = malloc_m(m, &m->w1t, 128 * 48)) ||
        (rc = malloc_m(m, &m->w2t, 128 * 128)) || (rc = malloc_m(m, &m->w3t, 16 * 128)) ||
        (rc = malloc_m(m, &m->w2r, 128 * 128)) || (rc = malloc_m(m, &m->w3r, 128 * 16)) ||
        (rc = malloc_m(m, &m->X, R * 48)) || (rc = malloc_m(m, &m->T, R * 3)) ||
        (rc = malloc_m(m, &m->Y, R * 3)) ||
        (rc = malloc_m(m, &m->rbuf, akmc_mlp_rows_bytes((int)R))) ||
        (rc = malloc_m(m, &m->P, (size_t)akmc_mlp_grad_chunks((int)R) * NP)) ||
        (rc = malloc_m(m, &m->lpart, akmc_mlp_grad_chunks((int)R))) || (rc = malloc_m(m, &m->ms, 96)))
        return bad(rc);
    HIPCHK(hipMemset(m->m1, 0, NP * sizeof(float)));
    HIPCHK(hipMemset(m->m2, 0, NP * sizeof(float)));
    // He-style initial weights from a seeded generator, zero biases
    std::vector<float> h(NP, 0.0f);
    unsigned long long st = 0x9E3779B97F4A7C15ull ^ seed;
    auto unif = [&]() {
        st += 0x9E3779B97F4A7C15ull;
        unsigned long long z = st;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return ((z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    };
    auto gauss = [&]() { return std::sqrt(-2.0 * std::log(unif())) * std::cos(6.283185307179586 * unif()); };
    size_t o = 0;
    for (int i = 0; i < 48 * 128; ++i) h[o++] = (float)(gauss() * std::sqrt(2.0 / 48));
    o += 128;
    for (int i = 0; i < 128 * 128; ++i) h[o++] = (float)(gauss() * std::sqrt(2.0 / 128));
    o += 128;
    for (int i = 0; i < 128 * 3; ++i) h[o++] = (float)(gauss() * std::sqrt(1.0 / 128));
    HIPCHK(hipMemcpy(m->p, h.data(), NP * sizeof(float), hipMemcpyHostToDevice));
    if ((rc = mlp_refresh_weights(m))) return bad(rc);
    HIPCHK(hipStreamSynchronize(m->stream));
    *out = m;
    return AKMC_SUCCESS;
}

void akmc_mlp_destroy(akmc_mlp_t m) { mlp_free(m); }

int akmc_mlp_set_params(akmc_mlp_t m, const float *params)
{
    if (!m || !params) return fail(AKMC_EINVAL, "bad arguments");
    HIPCHK(hipMemcpyAsync(m->p, params, AKMC_MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice, m->stream));
    TRY(mlp_refresh_weights(m));
    HIPCHK(hipStreamSynchronize(m->stream));
    return AKMC_SUCCESS;
}

int akmc_mlp_get_params(akmc_mlp_t m, float *params)
{
    if (!m || !params) return fail(AKMC_EINVAL, "bad arguments");
    HIPCHK(hipMemcpyAsync(params, m->p, AKMC_MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    return AKMC_SUCCESS;
}

int akmc_mlp_forward(akmc_mlp_t m, const float *X, int M, float *Y)
{
    return akmc_mlp_forward_scaled(m, X, nullptr, nullptr, M, Y);
}

int akmc_mlp_forward_scaled(akmc_mlp_t m, const float *X, const float *mean, const float *scale, int M, float *Y)
{
    if (!m || !X || !Y || M < 0 || !mean != !scale) return fail(AKMC_EINVAL, "bad arguments");
    // a few rows are standardised here: two more copies and a launch take
    // longer than their arithmetic (1 row 38 us so, 45 us on the device, 1024
    // rows 53 and 63 us)
    constexpr int kHostRows = 1024;
    std::vector<float> few;
    if (mean && M <= kHostRows) {
        few.resize((size_t)M * 48);
        for (int r = 0; r < M; ++r)
            for (int c = 0; c < 48; ++c) few[(size_t)r * 48 + c] = (X[(size_t)r * 48 + c] - mean[c]) * scale[c];
        X = few.data();
        mean = scale = nullptr;
    }
    TRY(mlp_scaling(m, mean, scale));
    for (int r0 = 0; r0 < M; r0 += m->rows) {
        int n = std::min(m->rows, M - r0);
        HIPCHK(hipMemcpyAsync(m->X, X + (size_t)r0 * 48, (size_t)n * 48 * sizeof(float), hipMemcpyHostToDevice,
                              m->stream));
        if (mean) akmc_mlp_launch_standardize(m->X, n, m->ms, m->ms + 48, m->stream);
        akmc_mlp_launch_forward(m->X, n, m->p, m->w1t, m->w2t, m->w3t, m->Y, m->stream);
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpyAsync(Y + (size_t)r0 * 3, m->Y, (size_t)n * 3 * sizeof(float), hipMemcpyDeviceToHost,
                              m->stream));
    }
    HIPCHK(hipStreamSynchronize(m->stream));
    return AKMC_SUCCESS;
}

int akmc_mlp_loss_grad(akmc_mlp_t m, const float *X, const float *T, int M, double *loss, float *grad)
{
    if (!m || !X || !T || M <= 0 || M > m->rows) return fail(AKMC_EINVAL, "M must be in [1, max_rows]");
    HIPCHK(hipMemcpyAsync(m->X, X, (size_t)M * 48 * sizeof(float), hipMemcpyHostToDevice, m->stream));
    HIPCHK(hipMemcpyAsync(m->T, T, (size_t)M * 3 * sizeof(float), hipMemcpyHostToDevice, m->stream));
    TRY(mlp_grad(m, m->X, m->T, nullptr, M, 0, 0.0f, nullptr));
    std::vector<double> part(akmc_mlp_grad_chunks(M));
    if (loss)
        HIPCHK(hipMemcpyAsync(part.data(), m->lpart, part.size() * sizeof(double), hipMemcpyDeviceToHost, m->stream));
    if (grad) HIPCHK(hipMemcpyAsync(grad, m->g, AKMC_MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    if (loss) {
        double s = 0.0;
        for (double v : part) s += v;
        *loss = s / M;
    }
    return AKMC_SUCCESS;
}

int akmc_mlp_time(akmc_mlp_t m, int M, int nrep, double ms[2])
{
    if (!m || !ms || M <= 0 || M > m->rows || nrep <= 0) return fail(AKMC_EINVAL, "M must be in [1, max_rows]");
    HIPCHK(hipMemsetAsync(m->X, 0, (size_t)M * 48 * sizeof(float), m->stream));
    HIPCHK(hipMemsetAsync(m->T, 0, (size_t)M * 3 * sizeof(float), m->stream));
    hipEvent_t e[3];
    for (auto &v : e) HIPCHK(hipEventCreate(&v));
    TRY(mlp_grad(m, m->X, m->T, nullptr, M, 0, 0.0f, nullptr));  // first launches outside the timing
    akmc_mlp_launch_forward(m->X, M, m->p, m->w1t, m->w2t, m->w3t, m->Y, m->stream);
    HIPCHK(hipEventRecord(e[0], m->stream));
    for (int r = 0; r < nrep; ++r)
        akmc_mlp_launch_forward(m->X, M, m->p, m->w1t, m->w2t, m->w3t, m->Y, m->stream);
    HIPCHK(hipEventRecord(e[1], m->stream));
    for (int r = 0; r < nrep; ++r) TRY(mlp_grad(m, m->X, m->T, nullptr, M, 0, 0.0f, nullptr));
    HIPCHK(hipEventRecord(e[2], m->stream));
    HIPCHK(hipEventSynchronize(e[2]));
    float t0 = 0.0f, t1 = 0.0f;
    HIPCHK(hipEventElapsedTime(&t0, e[0], e[1]));
    HIPCHK(hipEventElapsedTime(&t1, e[1], e[2]));
    for (auto &v : e) (void)hipEventDestroy(v);
    ms[0] = t0 / nrep;
    ms[1] = t1 / nrep;
    return AKMC_SUCCESS;
}

int akmc_mlp_train(akmc_mlp_t m, const float *X, const float *T, int M, int epochs, int batch, float lr,
                   unsigned seed, double *loss_history)
{
    return akmc_mlp_train_scaled(m, X, nullptr, nullptr, T, M, epochs, batch, lr, seed, loss_history);
}

int akmc_mlp_train_scaled(akmc_mlp_t m, const float *X, const float *mean, const float *scale, const float *T, int M,
                          int epochs, int batch, float lr, unsigned seed, double *loss_history)
{
    if (!m || !X || !T || M <= 0 || epochs <= 0 || batch <= 0 || batch > m->rows || !mean != !scale)
        return fail(AKMC_EINVAL, "bad training arguments (batch must be <= max_rows)");
    TRY(mlp_scaling(m, mean, scale));
    float *dX = nullptr, *dT = nullptr;
    int *didx = nullptr;
    hipEvent_t copied = nullptr;  // the permutation has left host memory
    double *dacc = nullptr;  // per-epoch loss accumulator (no host sync per minibatch)
    HIPCHK(hipMalloc(&dX, (size_t)M * 48 * sizeof(float)));
    HIPCHK(hipMalloc(&dT, (size_t)M * 3 * sizeof(float)));
    HIPCHK(hipMalloc(&didx, (size_t)M * sizeof(int)));
    HIPCHK(hipMalloc(&dacc, (size_t)epochs * sizeof(double)));
    HIPCHK(hipMemset(dacc, 0, (size_t)epochs * sizeof(double)));
    auto cleanup = [&]() {
        (void)hipFree(dX);
        (void)hipFree(dT);
        (void)hipFree(didx);
        (void)hipFree(dacc);
        if (copied) (void)hipEventDestroy(copied);
    };
    if (hipEventCreateWithFlags(&copied, hipEventDisableTiming) != hipSuccess) {
        copied = nullptr;
        cleanup();
        return fail(AKMC_EHIP, "event creation failed");
    }
    if (hipMemcpy(dX, X, (size_t)M * 48 * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dT, T, (size_t)M * 3 * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) {
        cleanup();
        return fail(AKMC_EHIP, "training data upload failed");
    }
    if (mean) {
        akmc_mlp_launch_standardize(dX, M, m->ms, m->ms + 48, m->stream);
        const hipError_t es = hipGetLastError();
        if (es != hipSuccess) {
            cleanup();
            return fail(AKMC_EHIP, "standardisation: %s", hipGetErrorString(es));
        }
    }
    std::vector<int> perm(M);
    unsigned long long st = 0xD1B54A32D192ED03ull ^ seed;
    auto next = [&]() {
        st += 0x9E3779B97F4A7C15ull;
        unsigned long long z = st;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    auto shuffle = [&]() {
        for (int i = 0; i < M; ++i) perm[i] = i;
        for (int i = M - 1; i > 0; --i) std::swap(perm[i], perm[next() % (unsigned long long)(i + 1)]);
    };
    int nbatch_ep = 1;
    shuffle();
    for (int ep = 0; ep < epochs; ++ep) {
        if (hipMemcpyAsync(didx, perm.data(), (size_t)M * sizeof(int), hipMemcpyHostToDevice, m->stream) !=
                hipSuccess ||
            hipEventRecord(copied, m->stream) != hipSuccess) {
            cleanup();
            return fail(AKMC_EHIP, "permutation upload failed");
        }
        int nb = 0;
        for (int b0 = 0; b0 + batch <= M || (b0 == 0 && M < batch); b0 += batch) {
            const int rc = mlp_grad(m, dX, dT, didx + b0, std::min(batch, M - b0), 1, lr, dacc + ep);
            if (rc != AKMC_SUCCESS) {
                cleanup();
                return rc;
            }
            ++nb;
            if (M < batch) break;
        }
        nbatch_ep = std::max(nb, 1);
        // the next epoch's order while this one trains
        if (ep + 1 < epochs) {
            if (hipEventSynchronize(copied) != hipSuccess) {
                cleanup();
                return fail(AKMC_EHIP, "training step failed");
            }
            shuffle();
        }
    }
    std::vector<double> acc(epochs);
    hipError_t e = hipMemcpyAsync(acc.data(), dacc, (size_t)epochs * sizeof(double), hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    cleanup();
    if (e != hipSuccess) return fail(AKMC_EHIP, "training failed: %s", hipGetErrorString(e));
    if (loss_history)
        for (int ep = 0; ep < epochs; ++ep) loss_history[ep] = acc[ep] / nbatch_ep;
    return AKMC_SUCCESS;
}

int akmc_batch_descriptors(akmc_batch_t b, int nq, const int *atom, const double *vac, const double *mover,
                           float *X)
{
    if (!b || nq <= 0 || !atom || !vac || !mover || !X) return fail(AKMC_EINVAL, "bad arguments");
    for (int q = 0; q < nq; ++q)
        if (atom[q] < 0 || atom[q] >= b->A) return fail(AKMC_EINVAL, "query %d: atom out of range", q);
    // the distinct atoms, in the order they are first asked for
    std::vector<int> slot_of(b->A, -1), uniq, ids(2 * (size_t)nq);
    for (int q = 0; q < nq; ++q) {
        int &sl = slot_of[atom[q]];
        if (sl < 0) {
            sl = (int)uniq.size();
            uniq.push_back(atom[q]);
        }
        ids[q] = atom[q];
        ids[nq + q] = sl;
    }
    const size_t n = nq, na = uniq.size();
    // one buffer of the batch: sites, movers, rows, atom terms, indices
    const size_t bytes = 48 * n + 192 * n + 128 * na + 8 * n + 4 * na;
    if (bytes > b->desc_n) {
        if (b->desc_dev) HIPCHK(hipFree(b->desc_dev));
        b->desc_dev = nullptr;
        b->desc_n = 0;
        HIPCHK(hipMalloc((void **)&b->desc_dev, bytes));
        b->desc_n = bytes;
    }
    double *qv = (double *)b->desc_dev, *qm = qv + 3 * n;
    float *qx = (float *)(qm + 3 * n), *G = qx + 48 * n;
    int *qi = (int *)(G + 32 * na), *ua = qi + 2 * n;
    HIPCHK(hipMemcpyAsync(qv, vac, 3 * n * sizeof(double), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(qm, mover, 3 * n * sizeof(double), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(qi, ids.data(), 2 * n * sizeof(int), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(ua, uniq.data(), na * sizeof(int), hipMemcpyHostToDevice, b->stream));
    akmc_mlp_launch_descriptors(b->d, (int)na, ua, nq, qi, qi + n, qv, qm, G, qx, b->stream);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(X, qx, 48 * n * sizeof(float), hipMemcpyDeviceToHost, b->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
    if (e != hipSuccess) return fail(AKMC_EHIP, "descriptors: %s", hipGetErrorString(e));
    // an overflow of an earlier force call has been reported there
    return b->d.maxnb > AKMC_DESC_CAP ? check_overflow(b) : AKMC_SUCCESS;
}

}  // extern "C"
