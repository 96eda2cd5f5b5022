// lbm_capi.cpp -- implementation of include/lbm_capi.h (host side; kernels live in *.hip).
//
// The context owns every device allocation and one non-blocking HIP stream (default
// priority).  The reference's set-up (System::System + LBM::LBM + LBM::Initialize,
// 3D MPI+KOKKOS+MPIIO/System.cpp:5-23, lbm.hpp:146-219, lbm.cpp:36-256) becomes
// lbm_create + lbm_initialize; its time loop body becomes lbm_step.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "internal.hpp"
#include "lattice.hpp"

using namespace lbm;

static thread_local std::string t_create_err;

static bool ref_mode(int bc) { return bc == LBM_BC_REFERENCE || bc == LBM_BC_REFERENCE_SN; }

static int set_err(lbm_ctx *c, int code, const std::string &m) {
    if (c) c->err = m;
    else t_create_err = m;
    return code;
}

#define HIP_TRY(c, expr)                                                                               \
    do {                                                                                               \
        hipError_t e__ = (expr);                                                                       \
        if (e__ != hipSuccess)                                                                         \
            return set_err((c), LBM_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e__));     \
    } while (0)

template <int Q>
static void table(int *e, double *w, int *opp) {
    static_for<0, Q>([&](auto I) {
        constexpr int i = I;
        if (e) {
            e[3 * i] = Lat<Q>::ex(i);
            e[3 * i + 1] = Lat<Q>::ey(i);
            e[3 * i + 2] = Lat<Q>::ez(i);
        }
        if (w) w[i] = Lat<Q>::w(i);
        if (opp) opp[i] = Lat<Q>::opp(i);
    });
}

extern "C" int lbm_lattice_table(int lattice, int *e, double *w, int *opp) {
    if (lattice == 9) table<9>(e, w, opp);
    else if (lattice == 27) table<27>(e, w, opp);
    else return LBM_ERR_INVALID;
    return LBM_OK;
}

extern "C" int lbm_config_default(lbm_config *c, int lattice) {
    if (!c || (lattice != 9 && lattice != 27)) return LBM_ERR_INVALID;
    std::memset(c, 0, sizeof(*c));
    const double cs2 = 1.0 / 3.0;
    c->lattice = lattice;
    c->rho0 = 1.0;
    c->precision = LBM_FP64;
    c->bc_mode = LBM_BC_REFERENCE;
    c->body = LBM_BODY_SPHERE;
    c->inlet = LBM_INLET_UNIFORM;
    c->seed = 5374857ull;   // the reference's Random_XorShift64_Pool seed
    if (lattice == 27) {
        // input.in: rho R Re / u0 Time inter / nx ny nz = 1.0 8.0 100 / 0.1 .. / 512 128 128
        const double R = 8.0, Re = 100.0;
        c->nx = 512; c->ny = 128; c->nz = 128;
        c->u0 = 0.1;
        c->tau0 = c->u0 * R / Re / cs2;                       // System.cpp:19
        c->cx = c->cy = c->cz = (double)((c->nx - 1) / 8);    // lbm.cpp:238 (integer division)
        const double r = (c->nx - 1) / 64.0;
        c->r2 = r * r;
        c->force_interval = 0;                                // the 3D reference logs no force
    } else {
        // MPI Kokkos/System.cpp:9-17 and main.cpp:8-9: nx 512, ny 128, R = int(0.1*ny)
        c->nx = 512; c->ny = 128; c->nz = 1;
        c->u0 = 0.1;
        const int R = (int)(0.1 * c->ny);
        c->tau0 = c->u0 * R / 100.0 / cs2;
        c->cx = 0.5 * (c->nx - 1);                            // lbm.cpp:108
        c->cy = 0.5 * (c->ny - 1);
        const double r = 0.03125 * (c->nx - 1) / 2.0;
        c->r2 = r * r;
        c->force_interval = 1;                                // test.dat every step, lbm.cpp:398-407
    }
    return LBM_OK;
}

extern "C" const char *lbm_last_error(const lbm_ctx *ctx) { return ctx ? ctx->err.c_str() : t_create_err.c_str(); }

static void free_all(lbm_ctx *c) {
    void *ptrs[] = {c->A, c->B, c->flags, c->dsfrac, c->duin, c->macros, c->block_slot, c->partials, c->hist, c->fix,
                    c->fixlk, c->rowwin, c->wlk, c->link, c->linklk, c->link_slot, c->rowclean, c->rf, c->rft, c->rmac, c->rprof, c->rusr, c->rfpre, c->rsurf,
                    c->snap_dev, c->dbad, c->tb_partials, c->tb_lk, c->rone.special, c->rone.rows, c->rone.links};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    c->A = c->B = nullptr;
    c->flags = nullptr;
    c->dsfrac = nullptr;
    c->duin = c->macros = c->partials = c->hist = nullptr;
    c->block_slot = nullptr;
    c->fix = c->fixlk = nullptr;
    c->rowwin = nullptr;
    c->wlk = nullptr;
    c->link = c->linklk = nullptr;
    c->link_slot = nullptr;
    c->rowclean = nullptr;
    c->nfix = c->nlink = 0;
    c->snap_dev = nullptr;
    c->dbad = nullptr;
    c->tb_partials = nullptr;
    c->tb_lk = nullptr;
    c->tb_k = 0;
    c->strip = false;
    c->rf = c->rft = c->rmac = c->rprof = c->rfpre = nullptr;
    c->rsurf = nullptr;
    c->nsurf = 0;
    c->rusr = nullptr;
    c->rone = RefOne{};
    pair_free(c->pair);
    output_free(c);
    if (c->snap_host) (void)hipHostFree(c->snap_host);
    c->snap_host = nullptr;
    c->snap_elems = 0;
}

extern "C" int lbm_create(const lbm_config *cfg, lbm_ctx **out) {
    if (!cfg || !out) return set_err(nullptr, LBM_ERR_INVALID, "null argument");
    *out = nullptr;
    const int Q = cfg->lattice;
    if (Q != 9 && Q != 27) return set_err(nullptr, LBM_ERR_INVALID, "lattice must be 9 (D2Q9) or 27 (D3Q27)");
    const int nz = Q == 9 ? 1 : cfg->nz;
    if (cfg->nx < 3 || cfg->ny < 3 || (Q == 27 && nz < 3) || (Q == 9 && cfg->nz > 1))
        return set_err(nullptr, LBM_ERR_INVALID, "extents: need nx, ny (and nz for D3Q27) >= 3, nz = 1 for D2Q9");
    if (!(cfg->tau0 > 0.0) || !std::isfinite(cfg->tau0))
        return set_err(nullptr, LBM_ERR_INVALID, "tau0 must be > 0 (relaxation time tau0 + 0.5 > 0.5)");
    if (cfg->precision < LBM_FP64 || cfg->precision > LBM_BF16S)
        return set_err(nullptr, LBM_ERR_INVALID, "unknown precision");
    if (!ref_mode(cfg->bc_mode) && cfg->bc_mode != LBM_BC_PLAIN)
        return set_err(nullptr, LBM_ERR_INVALID, "unknown bc_mode");
    if (cfg->bc_mode == LBM_BC_REFERENCE_SN && Q != 9)
        return set_err(nullptr, LBM_ERR_INVALID, "LBM_BC_REFERENCE_SN is the single-node 2D variant: lattice 9 only");
    if (ref_mode(cfg->bc_mode) && cfg->precision != LBM_FP64)
        return set_err(nullptr, LBM_ERR_INVALID, "reference boundary mode runs in FP64 only");
    if (cfg->body < LBM_BODY_NONE || cfg->body > LBM_BODY_MASK)
        return set_err(nullptr, LBM_ERR_INVALID, "unknown body");
    if (ref_mode(cfg->bc_mode) && cfg->body == LBM_BODY_MASK)
        return set_err(nullptr, LBM_ERR_INVALID, "reference mode takes its body from the sphere/cylinder formula");
    if (cfg->inlet < LBM_INLET_UNIFORM || cfg->inlet > LBM_INLET_PROFILE)
        return set_err(nullptr, LBM_ERR_INVALID, "unknown inlet");
    if (cfg->ncoef < 0 || cfg->ncoef > 8) return set_err(nullptr, LBM_ERR_INVALID, "ncoef must be in [0, 8]");
    if (cfg->force_interval < 0) return set_err(nullptr, LBM_ERR_INVALID, "force_interval must be >= 0");
    const int nxp = (cfg->nx + 63) / 64 * 64;
    const size_t plane = (size_t)nxp * cfg->ny * nz;
    if (plane >= (size_t)1 << 32) return set_err(nullptr, LBM_ERR_INVALID, "domain too large: the padded node count nxp*ny*nz must stay below 2^32");

    lbm_ctx *c = new lbm_ctx();
    c->cfg = *cfg;
    c->cfg.nz = nz;
    c->Q = Q;
    c->D = Q == 9 ? 2 : 3;
    c->prec = cfg->precision;
    c->geo.nx = cfg->nx;
    c->geo.ny = cfg->ny;
    c->geo.nz = nz;
    c->geo.nxp = nxp;
    c->geo.plane = plane;
    // populations row-interleaved (the Q direction rows of a row side by side); the layout with
    // one plane per direction (LBM_DIRECTION_PLANES) is kept for comparison, same results
    const bool planes = std::getenv("LBM_DIRECTION_PLANES") != nullptr;
    c->geo.ds = planes ? plane : (size_t)nxp;
    c->geo.rs = planes ? (size_t)nxp : (size_t)Q * nxp;
    const bool plain = cfg->bc_mode == LBM_BC_PLAIN;
    c->geo.xper = plain && cfg->periodic[0];
    c->geo.yper = plain && cfg->periodic[1];
    c->geo.zper = plain && Q == 27 && cfg->periodic[2];
    c->N = (size_t)cfg->nx * cfg->ny * nz;
    // nodes per lane of the fused kernel: one 4-byte access per direction for two FP16/BF16
    // nodes; FP32 and FP64 keep one node per lane (measured fastest on the 512x256x256 case).
    // LBM_NODES_PER_LANE overrides it among the instantiated widths (FP32: 1, 2; FP16/BF16: 2, 4).
    c->V = (c->prec == LBM_FP16S || c->prec == LBM_BF16S) ? 2 : 1;
    if (const char *env = std::getenv("LBM_NODES_PER_LANE")) {
        const int v = std::atoi(env);
        const bool ok = c->prec == LBM_FP32 ? (v == 1 || v == 2) : c->prec != LBM_FP64 && (v == 2 || v == 4);
        if (ok) c->V = v;
    }
    // 16-bit storage with two nodes per lane pulls with one (2-byte aligned) dword load per
    // direction; LBM_ALIGNED_PULL selects aligned loads with lane shifts instead (same
    // results; faster with one plane per direction, slower with the row-interleaved layout).
    c->aligned_pull = std::getenv("LBM_ALIGNED_PULL") != nullptr;
    // Blocks of the packed kernel resident per CU (256-lane blocks, row-interleaved populations).
    // D3Q27, measured on the 512x256x256 cylinder: FP32 fastest at 3 (3 waves per SIMD: 71.5 %
    // of HBM peak per step against 70.8 % uncapped), FP16/BF16 at 5 (steps 6-25 of the seeded
    // start: 0.647 ms per step against 0.664 at 4 and 0.649 at 6; later steps equal at 4 and 5).
    // D2Q9, measured on an 8192x4096 disk: FP32 fastest uncapped (78.5 % against 69.3 % at 3),
    // FP16/BF16 at 6 (73.5 % against 71.7 % uncapped and 67.4 % at 4).  The cap is a dynamic LDS
    // allocation the kernel does not use.  LBM_FAST_BLOCKS_PER_CU overrides it (0: no cap).
    // Rows of fewer than 256 lanes (narrow domains) keep the same waves per CU.
    // Reference mode's fused kernel (FP64, D3Q27): fastest at 3 (512x128x128 sphere: 0.730 ms per
    // step against 0.767 uncapped, 0.761 at 2, 0.751 at 4); the plain FP64 kernel gains nothing
    // (0.628-0.630 ms at none, 3, 4; 0.701 at 2), so it stays uncapped.
    int bpc = 0;
    if (c->prec == LBM_FP32) bpc = Q == 27 ? 3 : 0;
    else if (c->prec != LBM_FP64) bpc = Q == 27 ? 5 : 6;
    else if (ref_mode(cfg->bc_mode) && Q == 27) bpc = 3;
    if (const char *env = std::getenv("LBM_FAST_BLOCKS_PER_CU")) bpc = std::max(0, std::atoi(env));
    hipError_t e = hipSuccess;
    if (bpc > 0) {
        int dev = 0, lds = 0;
        e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev);
        if (e != hipSuccess) {
            set_err(nullptr, LBM_ERR_HIP, std::string("hipDeviceGetAttribute: ") + hipGetErrorString(e));
            delete c;
            return LBM_ERR_HIP;
        }
        // the count is of 4-wave (256-lane) blocks: rows narrower than 256 lanes launch smaller
        // blocks, and proportionally more of them may stay resident (the plain kernels); the
        // reference mode's fused kernel always launches 256-lane blocks
        const int lanes = ref_mode(cfg->bc_mode) ? 256 : nxp / c->V, wpb = (std::min(lanes, 256) + 63) / 64;
        const int blocks = std::max(1, bpc * 4 / wpb);
        // midway between lds/(blocks+1) and lds/blocks, so allocation granularity cannot tip the count
        const unsigned per = (unsigned)(2LL * lds / (2 * blocks + 1)) / 512u * 512u;
        if (per > (unsigned)lds / (unsigned)(blocks + 1) && per <= 65536u) c->fast_lds = per;
    }
    e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        set_err(nullptr, LBM_ERR_HIP, std::string("hipStreamCreateWithFlags: ") + hipGetErrorString(e));
        delete c;
        return LBM_ERR_HIP;
    }
    // lbm_get_fields_noalloc's staging array on this device (its own error, reported by that call)
    if (noalloc_setup(&c->noalloc_scratch, c->noalloc_err) != LBM_OK) c->noalloc_scratch = nullptr;
    *out = c;
    return LBM_OK;
}

int snapshot_wait(lbm_ctx *c);

extern "C" void lbm_destroy(lbm_ctx *c) {
    if (!c) return;
    snapshot_wait(c);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    free_all(c);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

extern "C" int lbm_set_mask(lbm_ctx *c, const uint8_t *solid) {
    if (!c || !solid) return set_err(c, LBM_ERR_INVALID, "null argument");
    if (c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_set_mask after lbm_initialize");
    if (c->cfg.body != LBM_BODY_MASK) return set_err(c, LBM_ERR_INVALID, "lbm_set_mask requires body = LBM_BODY_MASK");
    c->solid.assign(solid, solid + c->N);
    return LBM_OK;
}

extern "C" int lbm_set_solid_fraction(lbm_ctx *c, const double *s) {
    if (!c || !s) return set_err(c, LBM_ERR_INVALID, "null argument");
    if (c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_set_solid_fraction after lbm_initialize");
    if (c->cfg.bc_mode != LBM_BC_PLAIN) return set_err(c, LBM_ERR_INVALID, "partial bounce-back is a plain-mode feature");
    for (size_t n = 0; n < c->N; n++)
        if (!(s[n] >= 0.0 && s[n] <= 1.0)) return set_err(c, LBM_ERR_INVALID, "solid fraction outside [0, 1]");
    c->sfrac.assign(s, s + c->N);
    return LBM_OK;
}

extern "C" int lbm_set_inlet_profile(lbm_ctx *c, const double *uin) {
    if (!c || !uin) return set_err(c, LBM_ERR_INVALID, "null argument");
    if (c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_set_inlet_profile after lbm_initialize");
    c->uin.assign(uin, uin + (size_t)c->geo.ny * c->geo.nz);
    c->uin_set = true;
    return LBM_OK;
}

extern "C" int lbm_set_perturbation(lbm_ctx *c, const double *xi) {
    if (!c || !xi) return set_err(c, LBM_ERR_INVALID, "null argument");
    if (c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_set_perturbation after lbm_initialize");
    c->xi.assign(xi, xi + c->N);
    return LBM_OK;
}

static void ref_extents(const lbm_ctx *c, RefGeo &r) {
    r.Q = c->Q;
    r.D = c->D;
    r.g = c->D == 3 ? 3 : 2;   // ghost width: 3D MPI+KOKKOS+MPIIO/lbm.hpp:22, MPI Kokkos/lbm.hpp:79-80
    r.glx = c->geo.nx;
    r.gly = c->geo.ny;
    r.glz = c->geo.nz;
    r.lx = r.glx + 2 * r.g;
    r.ly = r.gly + 2 * r.g;
    r.lz = c->D == 3 ? r.glz + 2 * r.g : 1;
    // 3D rows padded to 32 doubles: a row of lx = nx + 6 doubles then starts on a 256-byte
    // boundary (about 15 % faster at nx = 512).  2D keeps px = lx, since its wall fills read
    // one column past a row end into the next row exactly as the reference's flat index does.
    r.px = c->D == 3 ? (r.lx + 31) / 32 * 32 : r.lx;
    r.plane = (size_t)r.px * r.ly * r.lz;
    // populations: 3D row-interleaved as in the plain path (every 3D access stays inside its
    // row: i +- 2 lies in [0, lx) at every node a fill, usrbc or pull touches), 2D one plane
    // per direction (the flat-index wrap above needs consecutive rows of one direction);
    // LBM_DIRECTION_PLANES selects planes in 3D too
    const bool planes = c->D == 2 || std::getenv("LBM_DIRECTION_PLANES") != nullptr;
    r.ds = planes ? r.plane : (size_t)r.px;
    r.rs = planes ? (size_t)r.px : (size_t)r.Q * r.px;
    r.tau0 = c->cfg.tau0;
    r.u0 = c->cfg.u0;
    r.variant = c->cfg.bc_mode == LBM_BC_REFERENCE_SN ? 1 : 0;
    r.lds = c->fast_lds;
}

extern "C" int lbm_set_ran(lbm_ctx *c, const int32_t *ran, size_t count) {
    if (!c || !ran) return set_err(c, LBM_ERR_INVALID, "null argument");
    if (c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_set_ran after lbm_initialize");
    if (!ref_mode(c->cfg.bc_mode)) return set_err(c, LBM_ERR_INVALID, "ran is the reference-mode perturbation");
    RefGeo r;
    ref_extents(c, r);
    if (count != (size_t)r.lx * r.ly * r.lz) return set_err(c, LBM_ERR_INVALID, "ran must cover the ghost-padded box lx*ly*lz");
    for (size_t n = 0; n < count; n++)
        if (ran[n] < 0 || ran[n] > 99) return set_err(c, LBM_ERR_INVALID, "ran values must lie in [0, 100)");
    c->ran.assign(ran, ran + count);
    return LBM_OK;
}

// ---- host-side geometry ----
static double legendre(int k, double x) {
    double p0 = 1.0, p1 = x;
    if (k == 0) return p0;
    for (int n = 1; n < k; n++) {
        const double p2 = ((2.0 * n + 1.0) * x * p1 - (double)n * p0) / (double)(n + 1);
        p0 = p1;
        p1 = p2;
    }
    return p1;
}

// inlet velocity u_x(y, z); walls sit half a spacing outside the first/last node
static void inlet_profile(const lbm_ctx *c, std::vector<double> &uin) {
    static const int LY[8] = {0, 1, 0, 2, 1, 0, 3, 0}, LZ[8] = {0, 0, 1, 0, 1, 2, 0, 3};
    const int ny = c->geo.ny, nz = c->geo.nz, D = c->D;
    uin.assign((size_t)ny * nz, 0.0);
    for (int z = 0; z < nz; z++)
        for (int y = 0; y < ny; y++) {
            const double ey = ((double)y + 0.5) / (double)ny, ez = ((double)z + 0.5) / (double)nz;
            const double by = 4.0 * ey * (1.0 - ey), bz = D == 3 ? 4.0 * ez * (1.0 - ez) : 1.0;
            double u;
            if (c->cfg.inlet == LBM_INLET_PARABOLIC) {
                u = c->cfg.u0 * by * bz;
            } else if (c->cfg.inlet == LBM_INLET_LEGENDRE) {
                double sum = 0.0;
                for (int k = 0; k < c->cfg.ncoef; k++) {
                    const double phi = D == 3 ? legendre(LY[k], 2.0 * ey - 1.0) * legendre(LZ[k], 2.0 * ez - 1.0)
                                              : legendre(k, 2.0 * ey - 1.0);
                    sum += c->cfg.coef[k] * phi;
                }
                u = by * bz * sum;
            } else {
                u = c->cfg.u0;
            }
            uin[y + (size_t)ny * z] = u;
        }
}

static int grow_hist(lbm_ctx *c, int need) {
    if (need <= c->hist_cap) return LBM_OK;
    int cap = std::max(need, std::max(1024, 2 * c->hist_cap));
    double *h = nullptr;
    HIP_TRY(c, hipMalloc(&h, (size_t)cap * 4 * sizeof(double)));
    if (c->hist) {
        HIP_TRY(c, hipMemcpyAsync(h, c->hist, (size_t)c->nrec * 4 * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
        HIP_TRY(c, hipStreamSynchronize(c->stream));
        (void)hipFree(c->hist);
    }
    c->hist = h;
    c->hist_cap = cap;
    return LBM_OK;
}

FusedArgs ctx_fused_args(const lbm_ctx *c) {
    FusedArgs a;
    std::memset(&a, 0, sizeof(a));
    a.g = c->geo;
    a.tau = c->cfg.tau0 + 0.5;
    a.rtau = 1.0 / a.tau;
    a.omega = (float)(1.0 / (c->cfg.tau0 + 0.5));
    // 16-bit formats: offset o_i = feq_i(0, (u_ref, 0, 0)) and o_i / w_i
    std::vector<int> e(3 * c->Q), opp(c->Q);
    std::vector<double> w(c->Q);
    lbm_lattice_table(c->Q, e.data(), w.data(), opp.data());
    const double U = c->cfg.store_uref;
    for (int i = 0; i < c->Q; i++) {
        const double eu = e[3 * i] * U;
        const double o = w[i] * (3.0 * eu + 4.5 * eu * eu - 1.5 * U * U);
        a.sp.off[i] = (float)o;
        a.sp.offw[i] = (float)(o / w[i]);
    }
    return a;
}

static int init_plain(lbm_ctx *c) {
    const Geo &g = c->geo;
    const int Q = c->Q;
    if (c->cfg.body == LBM_BODY_MASK && c->solid.size() != c->N)
        return set_err(c, LBM_ERR_STATE, "body = LBM_BODY_MASK needs lbm_set_mask first");
    if (!c->uin_set) inlet_profile(c, c->uin);
    std::vector<int> e(3 * Q), opp(Q);
    lbm_lattice_table(Q, e.data(), nullptr, opp.data());
    const int V = c->V;
    const bool sf = !c->sfrac.empty();
    const char *force_slow = std::getenv("LBM_FORCE_SLOW_PATH");
    const bool all_slow = c->prec != LBM_FP64 && force_slow && force_slow[0] == '1';
    const bool same_offsets = c->prec == LBM_FP64 || c->prec == LBM_FP32 || c->cfg.store_uref == 0.0;
    // node flags, solid fraction and the counts on the device (setup_kernels.hip): from the body formula
    // (the reference's "usr", 3D MPI+KOKKOS+MPIIO/lbm.cpp:238) or the user mask
    HIP_TRY(c, hipMalloc(&c->flags, g.plane));
    const Shape s1 = c->prec == LBM_FP64 ? fp64_shape(g, Q) : lane_shape(g, 1);
    // what the host reads of it comes back in one copy
    struct Counts {
        unsigned solid, near, fix;   // nodes of each kind, nodes of the fix list
    } counts;
    const size_t nblk = (size_t)s1.gx * g.ny * g.nz, nrow = (size_t)g.ny * g.nz, hold = sizeof(Counts) + nblk + nrow;
    std::vector<uint8_t> got(hold);
    {
        // the moment planes (32 bytes per padded node, 64 of them a row at least), which nothing uses yet,
        // hold the scratch: solid fraction, counts, force blocks, clean rows, mask
        HIP_TRY(c, hipMalloc(&c->macros, sizeof(double) * 4 * g.plane));
        const size_t fracb = sizeof(double) * c->N;
        double *const frac = sf ? c->macros : nullptr;
        uint8_t *const res = (uint8_t *)c->macros + fracb, *const mask = c->cfg.body == LBM_BODY_MASK ? res + hold : nullptr;
        if (mask) HIP_TRY(c, hipMemcpyAsync(mask, c->solid.data(), c->N, hipMemcpyHostToDevice, c->stream));
        if (sf) {
            HIP_TRY(c, hipMemcpyAsync(frac, c->sfrac.data(), sizeof(double) * c->N, hipMemcpyHostToDevice, c->stream));
            HIP_TRY(c, hipMalloc(&c->dsfrac, (c->prec == LBM_FP64 ? sizeof(double) : sizeof(float)) * g.plane));
            HIP_TRY(c, setup_sfrac(c->prec, frac, c->dsfrac, g, c->stream));
        }
        HIP_TRY(c, hipMalloc(&c->rowclean, nrow));
        const SetupBody body{c->cfg.body, c->cfg.cx, c->cfg.cy, c->cfg.cz, c->cfg.r2};
        const SetupFix fx{V, all_slow, same_offsets};
        HIP_TRY(c, setup_flags(Q, c->flags, mask, frac, body, fx, g, (unsigned *)res, c->stream));
        HIP_TRY(c, setup_forced(c->flags, frac, res + sizeof(Counts), s1, g, c->stream));
        HIP_TRY(c, setup_clean(c->flags, c->rowclean, res + sizeof(Counts) + nblk, g, c->stream));
        HIP_TRY(c, hipMemcpyAsync(got.data(), res, hold, hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(c, hipStreamSynchronize(c->stream));
    }
    std::memcpy(&counts, got.data(), sizeof(counts));
    const uint8_t *const forced_blk = got.data() + sizeof(Counts);   // per block of shape s1: holds a forced node
    uint8_t *const clean = got.data() + sizeof(Counts) + nblk;       // per row: all nodes fluid with no solid neighbour
    c->solid_nodes = (int)counts.solid;
    c->near_nodes = (int)counts.near;
    // Dense mode: one per-node pass over every node instead of the copies, the packed pass
    // and the fix-up of the list, chosen
    //  * when the fix list holds more than a quarter of the fluid nodes (a solid fraction
    //    over a noisy field: half of them on the 192x96x96 adjoint workload, where the
    //    list path took 67 + 100 us per step and the dense pass 67 us), or
    //  * when a population buffer is at most 16 MB: such steps are launch-bound, and one
    //    launch fewer per step counts (D2Q9 512x128 with the drag every step: 6.7 / 6.4 us
    //    per step in FP32 / FP16 against 8.7 / 8.8; on D3Q27 512x128x128 the dense pass
    //    is as fast in FP32 but 1.5 times slower in FP16, so large domains keep the list).
    // LBM_DENSE=1 / 0 forces the choice.
    if (c->prec != LBM_FP64) {
        const size_t pop_bytes = (size_t)(c->prec == LBM_FP32 ? 4 : 2) * Q * g.plane;
        const bool small = pop_bytes <= ((size_t)16 << 20);
        const char *dense_env = std::getenv("LBM_DENSE");
        c->dense = dense_env ? dense_env[0] == '1' : (!all_slow && ((size_t)counts.fix * 4 > c->N - counts.solid || small));
    }
    const bool per_block = c->prec == LBM_FP64 || c->dense;
    // the lists below are per node; a dense or FP64 step needs none
    std::vector<uint8_t> flags;
    std::vector<uint32_t> near_list;   // D3Q27: the nodes next to the mask
    if (!per_block) {
        flags.resize(g.plane);
        HIP_TRY(c, hipMemcpyAsync(flags.data(), c->flags, g.plane, hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(c, hipStreamSynchronize(c->stream));
    }
    auto solid_at = [&](int x, int y, int z) -> bool {
        if (g.xper) x = (x + g.nx) % g.nx;
        if (g.yper) y = (y + g.ny) % g.ny;
        if (g.zper) z = (z + g.nz) % g.nz;
        if (x < 0 || x >= g.nx || y < 0 || y >= g.ny || z < 0 || z >= g.nz) return false;
        return flags[(size_t)x + (size_t)g.nxp * ((size_t)y + (size_t)g.ny * z)] == FL_SOLID;
    };
    // per-node kernels over every node (FP64 k_fused, dense mode k_dense_v; one node per lane):
    // a force partial slot per block holding a forced node
    std::vector<int> slot;
    c->nslots = 0;
    if (per_block) {
        slot.resize(nblk);
        for (size_t b = 0; b < slot.size(); b++) slot[b] = forced_blk[b] ? c->nslots++ : -1;
    }
    // FP32/16-bit: per fluid node (row-major padded indices), either
    //  * the link list: mask neighbours whose half-way bounce-back the packed kernel applies
    //    in its pull, from per-row windows of link words and force slots (below), or
    //  * the fix list, recomputed per node after the packed path: nodes with a solid fraction,
    //    the periodic x edges, the last node when nx is not a multiple of the lane width V
    //    (its lane reaches into the padding), and mask neighbours in the inlet or outlet lane
    //    (whose packs the packed kernel shifts by one node) or, when opposite directions have
    //    different storage offsets (16-bit storage with store_uref != 0), every mask neighbour
    //    (the packed kernel substitutes stored values, not decoded ones).
    // LBM_FORCE_SLOW_PATH=1 puts every fluid node on the fix list.  Force partial slots go to
    // the forced nodes in node order across both lists, so the force sum does not depend on
    // which list a node is on.
    if (!per_block) {
        std::vector<uint32_t> fix, fixlk, link, linklk;
        std::vector<int> lslot;
        for (int z = 0; z < g.nz; z++)
            for (int y = 0; y < g.ny; y++) {
                if (!sf && !all_slow && !g.xper && g.nx % V == 0 && clean[(size_t)y + (size_t)g.ny * z]) continue;   // nothing listed
                for (int x = 0; x < g.nx; x++) {
                    const size_t node = (size_t)x + (size_t)g.nxp * ((size_t)y + (size_t)g.ny * z);
                    if (flags[node] == FL_SOLID) continue;
                    const bool near = flags[node] == FL_NEAR;
                    const bool sfr = sf && c->sfrac[(size_t)x + (size_t)g.nx * ((size_t)y + (size_t)g.ny * z)] > 0.0;
                    const bool f = near || sfr;   // a node whose links or solid fraction carry force
                    const bool to_fix = all_slow || sfr || fix_edge(g, V, x) || (near && (fix_end_lane(g, V, x) || !same_offsets));
                    if (!to_fix && !near) continue;
                    if (near && Q == 27) near_list.push_back((uint32_t)node);
                    // link word: the per-node pull's classification (Zou-He unknowns and wall
                    // links first, outlet clamp, periodic wrap), bit i when the source is solid
                    uint32_t bits = 0;
                    if (near)
                        for (int i = 1; i < Q; i++) {
                            const int ex = e[3 * i], ey = e[3 * i + 1], ez = e[3 * i + 2];
                            if (ex > 0 && x == 0 && !g.xper) continue;
                            int sx = x - ex;
                            const int sy = y - ey, sz = z - ez;
                            if ((sy < 0 || sy >= g.ny) && !g.yper) continue;
                            if ((sz < 0 || sz >= g.nz) && !g.zper) continue;
                            if (sx == g.nx && !g.xper) sx = g.nx - 1;
                            if (solid_at(sx, sy, sz)) bits |= 1u << i;
                        }
                    const int k = f ? c->nslots++ : -1;
                    if (to_fix) {
                        fix.push_back((uint32_t)node);
                        fixlk.push_back(bits);
                        slot.push_back(k);
                    } else {
                        link.push_back((uint32_t)node);
                        linklk.push_back(bits);
                        lslot.push_back(k);
                    }
                }
            }
        if (fix.size() > (size_t)INT32_MAX || link.size() > (size_t)INT32_MAX)
            return set_err(c, LBM_ERR_INVALID, "too many boundary nodes");
        c->nfix = (int)fix.size();
        c->nlink = (int)link.size();
        if (c->nfix) {
            HIP_TRY(c, hipMalloc(&c->fix, sizeof(uint32_t) * fix.size()));
            HIP_TRY(c, hipMemcpy(c->fix, fix.data(), sizeof(uint32_t) * fix.size(), hipMemcpyHostToDevice));
            HIP_TRY(c, hipMalloc(&c->fixlk, sizeof(uint32_t) * fixlk.size()));
            HIP_TRY(c, hipMemcpy(c->fixlk, fixlk.data(), sizeof(uint32_t) * fixlk.size(), hipMemcpyHostToDevice));
        }
        // Per-row windows of the link list for the packed kernel: row r's lanes [t0, t0 + nl)
        // cover its linked nodes; the window's nl*V nodes hold their link words (0 for nodes
        // without links) from element `base` of wlk.  The list itself serves force steps.
        if (c->nlink) {
            std::vector<int4> win((size_t)g.ny * g.nz, make_int4(0, 0, 0, 0));
            std::vector<uint32_t> wlk;
            for (size_t j = 0; j < link.size();) {
                const uint32_t row = link[j] / (uint32_t)g.nxp;
                size_t k = j;
                while (k < link.size() && link[k] / (uint32_t)g.nxp == row) k++;   // the row's entries (node order)
                const int t0 = (int)(link[j] - row * (uint32_t)g.nxp) / V;
                const int t1 = (int)(link[k - 1] - row * (uint32_t)g.nxp) / V;
                const size_t base = wlk.size();
                if (base + (size_t)(t1 - t0 + 1) * V > (size_t)INT32_MAX)
                    return set_err(c, LBM_ERR_INVALID, "too many mask links");
                wlk.resize(base + (size_t)(t1 - t0 + 1) * V, 0u);
                for (size_t m = j; m < k; m++)
                    wlk[base + (link[m] - row * (uint32_t)g.nxp) - (size_t)t0 * V] = linklk[m];
                win[row] = make_int4(t0, t1 - t0 + 1, (int)base, 0);
                j = k;
            }
            HIP_TRY(c, hipMalloc(&c->rowwin, sizeof(int4) * win.size()));
            HIP_TRY(c, hipMemcpy(c->rowwin, win.data(), sizeof(int4) * win.size(), hipMemcpyHostToDevice));
            HIP_TRY(c, hipMalloc(&c->wlk, sizeof(uint32_t) * wlk.size()));
            HIP_TRY(c, hipMemcpy(c->wlk, wlk.data(), sizeof(uint32_t) * wlk.size(), hipMemcpyHostToDevice));
            HIP_TRY(c, hipMalloc(&c->link, sizeof(uint32_t) * link.size()));
            HIP_TRY(c, hipMemcpy(c->link, link.data(), sizeof(uint32_t) * link.size(), hipMemcpyHostToDevice));
            HIP_TRY(c, hipMalloc(&c->linklk, sizeof(uint32_t) * linklk.size()));
            HIP_TRY(c, hipMemcpy(c->linklk, linklk.data(), sizeof(uint32_t) * linklk.size(), hipMemcpyHostToDevice));
            HIP_TRY(c, hipMalloc(&c->link_slot, sizeof(int) * lslot.size()));
            HIP_TRY(c, hipMemcpy(c->link_slot, lslot.data(), sizeof(int) * lslot.size(), hipMemcpyHostToDevice));
        }
    }
    // D2Q9 on a small domain, where a step costs about a dependent launch: several steps per launch
    // (temporal blocking, small_kernel.hpp), for walls, inlet, outlet, a mask and a solid fraction,
    // up to 420 000 nodes (padded), in FP32 330 000.  On larger ones, and where an axis is periodic,
    // STRIP_K steps per pass over memory (strip_kernel.hpp), from 360 000 nodes on, in FP32 from 330 000 and
    // in 16-bit storage from 3 million.  us per step with drag every 10 steps, one launch per step / tiles / strips
    // (in brackets tiles / strips with the drag every step, where the order changes):
    //               FP64                 FP32                            FP16
    //   600x150     5.76 / 2.54 / 7.4    4.68 / 1.65 / 5.2               4.47 / 1.73 / 5.5
    //   1000x250    9.80 / 6.22 / 11.0   6.38 / 3.67 / 6.1               5.64 / 3.99 / 6.5
    //   1200x300    12.0 / 9.32 / 11.2   7.84 / 6.26 / 6.2 (8.5 / 6.8)   6.82 / 6.48 / 6.6 (8.5 / 7.2)
    //   1400x350    15.8 / 12.7 / 12.3   9.26 / 5.92 / 7.3 (8.0 / 8.0)   8.28 / 5.48 / 8.3 (7.6 / 9.0)
    //   2000x500    27.3 / 21.6 / 16.4   15.1 / 18.7 / 9.1               9.99 / 16.7 / 11.2
    //   2048x2048   100 / - / 55.4       50.4 / - / 24.5                 27.0 / - / 25.1
    // LBM_TEMPORAL_BLOCKING=0 keeps one step per launch, 1 / 2 take the tiles / the strips
    // regardless of the size.
    {
        const char *tbe = std::getenv("LBM_TEMPORAL_BLOCKING");
        // (FP32/16-bit: not under a switch that selects among the one-step kernels, and only where
        // opposite directions share their storage offset, as a bounced value is taken as stored)
        bool eligible = Q == 9;
        if (c->prec != LBM_FP64) {
            for (const char *k : {"LBM_FORCE_SLOW_PATH", "LBM_DENSE", "LBM_ALIGNED_PULL", "LBM_NODES_PER_LANE", "LBM_FAST_BLOCKS_PER_CU"})
                eligible = eligible && std::getenv(k) == nullptr;
            eligible = eligible && (c->prec == LBM_FP32 || c->cfg.store_uref == 0.0);
        }
        const bool small = g.plane <= (c->prec == LBM_FP32 ? 330000u : 420000u), tiles_ok = eligible && !g.xper && !g.yper;
        const bool large = g.plane >= (c->prec == LBM_FP64 ? 360000u : c->prec == LBM_FP32 ? 330000u : 3000000u);
        const size_t esz9 = c->prec == LBM_FP64 ? 8 : c->prec == LBM_FP32 ? 4 : 2;
        int dev = 0, lds_max = 0;
        if (eligible && (hipGetDevice(&dev) != hipSuccess ||
                         hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
                         hipDeviceGetAttribute(&c->cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess))
            eligible = false;
        int nparts = 0, slots = 0;
        if (eligible && tiles_ok && (tbe ? tbe[0] == '1' : small)) {
            int K = 0, T = 0;
            tb_choose(g, c->prec, c->cfg.force_interval, c->cus, K, T);
            if (K > 0 && (size_t)lds_max >= tb_lds_bytes(c->prec, T) + 4096 + 512 &&
                tb_prepare(c->prec, T, sf ? c : nullptr, ctx_fused_args(c)) == hipSuccess) {
                c->tb_k = K;
                c->tb_t = T;
                int tiles_x = 0;
                nparts = tb_tiles(g, T, K, &tiles_x);
                slots = tb_records(K);
            }
        } else if (eligible && (tbe ? tbe[0] == '2' : large) && g.ds == (size_t)g.nxp && esz9 * Q * g.plane < ((size_t)1 << 32)) {
            // (byte offsets in 32 bits)
            c->strip = true;
            for (int k = 2; k <= STRIP_K; k++) {
                StripLaunch l{};
                strip_shape(g, c->prec, c->cus, k, l);
                nparts = std::max(nparts, l.nwaves);
            }
            slots = tb_records(STRIP_K);
        }
        if (nparts > 0) {
            HIP_TRY(c, hipMalloc(&c->tb_partials, sizeof(double) * 3 * (size_t)nparts * slots));
            HIP_TRY(c, hipMalloc(&c->tb_lk, sizeof(uint16_t) * g.plane));
            HIP_TRY(c, setup_links9(c->flags, c->tb_lk, g, c->stream));
        }
    }
    const size_t esz = c->prec == LBM_FP64 ? 8 : c->prec == LBM_FP32 ? 4 : 2;
    HIP_TRY(c, hipMalloc(&c->A, esz * Q * g.plane));
    HIP_TRY(c, hipMalloc(&c->B, esz * Q * g.plane));
    HIP_TRY(c, hipMalloc(&c->duin, sizeof(double) * c->uin.size()));
    HIP_TRY(c, hipMalloc(&c->block_slot, sizeof(int) * std::max<size_t>(slot.size(), 1)));
    HIP_TRY(c, hipMalloc(&c->partials, force_bytes(c->nslots)));
    // D3Q27: two steps per pass over memory where the two-step kernel applies (pair.cpp); its force
    // slots are those of the one-step path
    if (Q == 27) {
        HIP_TRY(c, pair_plan(c->pair, c->prec, g, c->flags, same_offsets, !per_block && c->nfix == 0, sf ? std::vector<uint32_t>() : near_list,
                             per_block && !sf ? slot : std::vector<int>(), s1, c->stream));
    }
    {
        // (the adjoint's straight-line rows; LBM_ADJ_GENERAL_PATH=1 sends every row through the general
        // path, for tests)
        if (std::getenv("LBM_ADJ_GENERAL_PATH")) {
            std::fill(clean, clean + nrow, (uint8_t)0);
            HIP_TRY(c, hipMemcpy(c->rowclean, clean, nrow, hipMemcpyHostToDevice));
        }
        c->adj_all_fast = true;
        for (int z = 0; z < g.nz; z++)
            for (int y = 0; y < g.ny; y++) {
                const bool pedge = (g.yper && (y == 0 || y == g.ny - 1)) || (Q == 27 && g.zper && (z == 0 || z == g.nz - 1));
                if (!clean[(size_t)y + (size_t)g.ny * z] || pedge) c->adj_all_fast = false;
            }
    }
    HIP_TRY(c, hipMemcpyAsync(c->duin, c->uin.data(), sizeof(double) * c->uin.size(), hipMemcpyHostToDevice, c->stream));
    if (!slot.empty())
        HIP_TRY(c, hipMemcpy(c->block_slot, slot.data(), sizeof(int) * slot.size(), hipMemcpyHostToDevice));
    double *dxi = nullptr;
    if (!c->xi.empty()) {
        HIP_TRY(c, hipMalloc(&dxi, sizeof(double) * c->N));
        HIP_TRY(c, hipMemcpyAsync(dxi, c->xi.data(), sizeof(double) * c->N, hipMemcpyHostToDevice, c->stream));
    }
    const FusedArgs a = ctx_fused_args(c);
    HIP_TRY(c, plain_init(Q, c->prec, c->A, c->B, c->macros, c->flags, c->duin, dxi, c->cfg.perturb, c->cfg.seed, a, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    if (dxi) (void)hipFree(dxi);
    return LBM_OK;
}

static int init_ref(lbm_ctx *c) {
    RefGeo &r = c->rg;
    ref_extents(c, r);
    const int Q = c->Q;
    HIP_TRY(c, hipMalloc(&c->rf, sizeof(double) * Q * r.plane));
    HIP_TRY(c, hipMalloc(&c->rft, sizeof(double) * Q * r.plane));
    HIP_TRY(c, hipMalloc(&c->rmac, sizeof(double) * 4 * r.plane));
    HIP_TRY(c, hipMalloc(&c->rusr, r.plane));
    HIP_TRY(c, hipMalloc(&c->rfpre, sizeof(double) * Q * r.plane));
    const int nprof = c->D == 3 ? r.glz : r.gly;
    std::vector<double> prof(nprof);
    for (int k = 0; k < nprof; k++)   // u0*4*c*(n-1-c)/(n-1)^2, lbm.cpp:405 / MPI Kokkos/lbm.cpp:446
        prof[k] = c->cfg.u0 * 4.0 * (double)k * (double)(nprof - 1 - k) / ((double)(nprof - 1) * (double)(nprof - 1));
    HIP_TRY(c, hipMalloc(&c->rprof, sizeof(double) * nprof));
    HIP_TRY(c, hipMemcpyAsync(c->rprof, prof.data(), sizeof(double) * nprof, hipMemcpyHostToDevice, c->stream));
    int32_t *dran = nullptr;
    if (!c->ran.empty()) {
        HIP_TRY(c, hipMalloc(&dran, sizeof(int32_t) * c->ran.size()));   // unpadded lx*ly*lz
        HIP_TRY(c, hipMemcpyAsync(dran, c->ran.data(), sizeof(int32_t) * c->ran.size(), hipMemcpyHostToDevice, c->stream));
    }
    HIP_TRY(c, ref_init(r, c->rf, c->rft, c->rmac, c->rusr, dran, c->cfg.body, c->cfg.cx, c->cfg.cy, c->cfg.cz,
                        c->cfg.r2, c->cfg.seed, c->stream));
    // before the first step the reference's f is the initial equilibrium
    HIP_TRY(c, hipMemcpyAsync(c->rfpre, c->rf, sizeof(double) * Q * r.plane, hipMemcpyDeviceToDevice, c->stream));
    std::vector<uint8_t> usr(r.plane);
    HIP_TRY(c, hipMemcpyAsync(usr.data(), c->rusr, r.plane, hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    if (dran) (void)hipFree(dran);
    // usrbc works in place; reject masks for which its result would depend on thread order
    // (a solid node, a fluid gap of one node and another solid node along a link)
    std::vector<int> e(3 * Q);
    lbm_lattice_table(Q, e.data(), nullptr, nullptr);
    const int g = r.g, klo = c->D == 3 ? g : 0, khi = c->D == 3 ? r.lz - g : 1;
    c->solid_nodes = 0;
    std::vector<uint32_t> surf;   // usrbc's work list: interior solid nodes with a fluid neighbour
    for (int k = klo; k < khi; k++)
        for (int j = g; j < r.ly - g; j++)
            for (int i = g; i < r.lx - g; i++) {
                const long n = i + (long)r.px * (j + (long)r.ly * k);
                if (usr[n] != 0) continue;
                c->solid_nodes++;
                bool wet = false;
                for (int q = 1; q < Q; q++) {
                    const long d = e[3 * q] + (long)r.px * (e[3 * q + 1] + (long)r.ly * e[3 * q + 2]);
                    if (usr[n + d] == 1 && usr[n + 2 * d] == 0)
                        return set_err(c, LBM_ERR_INVALID, "reference mode: body has a one-node fluid gap along a lattice link (usrbc would race)");
                    wet = wet || usr[n + d] == 1;
                }
                if (wet) surf.push_back((uint32_t)n);
            }
    // 3D only: the 2D box (65 536 nodes by default) is launch-bound, and its step measured 7 %
    // slower with the list than with the interior sweep
    if (c->D == 3 && r.plane <= UINT32_MAX) {
        c->nsurf = (int)surf.size();
        HIP_TRY(c, hipMalloc(&c->rsurf, sizeof(uint32_t) * std::max<size_t>(surf.size(), 1)));
        if (!surf.empty())
            HIP_TRY(c, hipMemcpy(c->rsurf, surf.data(), sizeof(uint32_t) * surf.size(), hipMemcpyHostToDevice));
    }
    // 2D: a whole step in one launch where the fills and usrbc can be resolved (one block sums the drag, so
    // up to 16 384 links)
    if (c->D == 2) {
        std::vector<int> special, rows;
        std::vector<RefLink> links;
        if (ref_resolve(r, usr, special, rows, links) && links.size() <= 16384) {
            HIP_TRY(c, hipMalloc(&c->rone.special, sizeof(int) * special.size()));
            HIP_TRY(c, hipMalloc(&c->rone.rows, sizeof(int) * std::max<size_t>(rows.size(), 1)));
            HIP_TRY(c, hipMalloc(&c->rone.links, sizeof(RefLink) * std::max<size_t>(links.size(), 1)));
            HIP_TRY(c, hipMemcpy(c->rone.special, special.data(), sizeof(int) * special.size(), hipMemcpyHostToDevice));
            HIP_TRY(c, hipMemcpy(c->rone.rows, rows.data(), sizeof(int) * rows.size(), hipMemcpyHostToDevice));
            if (!links.empty())
                HIP_TRY(c, hipMemcpy(c->rone.links, links.data(), sizeof(RefLink) * links.size(), hipMemcpyHostToDevice));
            c->rone.nlinks = (int)links.size();
            c->rone.on = true;
        }
    }
    const int nblk = ref_mem_blocks(r);
    HIP_TRY(c, hipMalloc(&c->partials, sizeof(double) * 3 * nblk));
    c->nslots = nblk;
    return LBM_OK;
}

extern "C" int lbm_initialize(lbm_ctx *c) {
    if (!c) return LBM_ERR_INVALID;
    if (c->initialized) return set_err(c, LBM_ERR_STATE, "already initialised");
    int rc = c->cfg.bc_mode == LBM_BC_PLAIN ? init_plain(c) : init_ref(c);
    if (rc == LBM_OK) {
        const hipError_t e = hipMalloc(&c->dbad, sizeof(unsigned));
        if (e != hipSuccess) rc = set_err(c, LBM_ERR_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
    }
    if (rc != LBM_OK) {
        free_all(c);
        return rc;
    }
    c->initialized = true;
    c->step = 0;
    c->stage = 0;
    c->nrec = c->nrec_checked = 0;
    c->fields_fresh = true;   // the initial macros
    c->replay_ok = false;
    return LBM_OK;
}

StepBufs step_bufs(const lbm_ctx *c, const void *A, void *B) {
    StepBufs b;
    b.A = A;
    b.B = B;
    b.flags = c->flags;
    b.fix = c->fix;
    b.fixlk = c->fixlk;
    b.nfix = c->nfix;
    b.rowwin = c->rowwin;
    b.wlk = c->wlk;
    b.link = c->link;
    b.linklk = c->linklk;
    b.link_slot = c->link_slot;
    b.nlink = c->nlink;
    b.sfrac = c->dsfrac;
    b.uin = c->duin;
    b.block_slot = c->block_slot;
    b.dense = c->dense;
    b.partials = c->partials;
    b.macros = c->macros;
    b.aligned_pull = c->aligned_pull;
    b.fast_lds = c->fast_lds;
    b.ev_bulk[0] = b.ev_bulk[1] = nullptr;
    return b;
}

// Reference mode, after the fills: usrbc and, on force steps, the momentum exchange.  In 2D
// (launch-bound, the drag every step by default) one pass does both; in 3D usrbc runs over its
// list and the exchange separately.
static hipError_t ref_boundary_pass(lbm_ctx *c, bool force) {
    if (force && c->rone.on) {
        const hipError_t e = ref_usrbc(c->rg, c->rf, c->rusr, c->rsurf, c->nsurf, c->stream);
        return e != hipSuccess ? e : ref_one_force(c->rg, c->rone, c->rf, c->hist, c->nrec++, c->step, c->stream);
    }
    if (force && c->D == 2)
        return ref_mem(c->rg, c->rf, c->rusr, c->partials, c->nslots, c->hist, c->nrec++, c->step, true, c->stream);
    hipError_t e = ref_usrbc(c->rg, c->rf, c->rusr, c->rsurf, c->nsurf, c->stream);
    if (e == hipSuccess && force)
        e = ref_mem(c->rg, c->rf, c->rusr, c->partials, c->nslots, c->hist, c->nrec++, c->step, false, c->stream);
    return e;
}

// evs: null, or 2n events recorded around each step's bulk kernel (plain mode)
static int step_n(lbm_ctx *c, int n, hipEvent_t *evs = nullptr) {
    if (c->stage != 0)
        return set_err(c, LBM_ERR_STATE, "a staged step is in progress: finish it with lbm_boundary, lbm_stream, lbm_update");
    const int fi = c->cfg.force_interval;
    const int nforce = fi > 0 ? (int)((c->step + n) / fi - c->step / fi) : 0;
    int rc = grow_hist(c, c->nrec + nforce + 1);
    if (rc != LBM_OK) return rc;
    if (ref_mode(c->cfg.bc_mode)) {
        for (int k = 0; k < n; k++) {
            c->step++;
            const bool force = fi > 0 && c->step % fi == 0;
            if (c->rone.on) {
                HIP_TRY(c, ref_one(c->rg, c->rone, c->rf, c->rft, nullptr, c->rusr, c->rprof, nullptr, force ? c->hist : nullptr,
                                   c->nrec, c->step, c->stream));
                c->nrec += force;
                std::swap(c->rf, c->rft);
                c->fields_fresh = false;
                c->replay_ok = true;
                continue;
            }
            HIP_TRY(c, ref_fills(c->rg, c->rf, c->rft, c->stream));
            HIP_TRY(c, ref_boundary_pass(c, force));
            HIP_TRY(c, ref_fused(c->rg, c->rf, c->rft, nullptr, c->rusr, c->rprof, nullptr, c->stream));
            std::swap(c->rf, c->rft);
            c->fields_fresh = false;
            c->replay_ok = true;
        }
        return LBM_OK;
    }
    const FusedArgs a = ctx_fused_args(c);
    // temporally blocked launches for all but the last step (which stays a one-step launch, so
    // its input buffer can serve the fields on request); not under per-kernel timing
    // (their force records are summed together, when the partials' slots are full and before the
    // one-step launches, which write records of their own)
    int left = n;
    int pend = 0, rec0 = 0;
    long step1 = 0;
    auto records = [&](long step) { return fi > 0 && step % fi == 0; };
    const int depth = c->tb_k > 0 ? c->tb_k : c->strip ? STRIP_K : 0, slots = tb_records(depth);
    int nparts = 0, tiles_x = 0;   // partials per record of the pending records
    if (c->tb_k > 0) nparts = tb_tiles(a.g, c->tb_t, c->tb_k, &tiles_x);
    while (depth > 0 && !evs && left > (c->strip ? 2 : 1)) {
        const int kk = std::min(depth, left - 1);
        StripLaunch l{};
        if (c->strip) strip_shape(a.g, c->prec, c->cus, kk, l);
        if (pend + kk > slots || (c->strip && pend > 0 && l.nwaves != nparts)) {
            HIP_TRY(c, tb_force_flush(c->tb_partials, nparts, slots, c->hist, rec0, pend, step1, fi, c->stream));
            pend = 0;
        }
        if (c->strip) nparts = l.nwaves;
        if (pend == 0 && fi > 0) {
            rec0 = c->nrec;
            step1 = (c->step + fi) / fi * fi;   // the first force step after the current one
        }
        int nr = 0;
        if (c->strip) {
            l.A = c->A;
            l.B = c->B;
            l.lk = c->tb_lk;
            l.sfrac = c->dsfrac;
            l.uin = c->duin;
            l.partials = c->tb_partials;
            l.pend = pend;
            for (int j = 0; j < kk; j++)
                if (records(c->step + j + 1)) {
                    l.rec |= 1u << j;
                    nr++;
                }
            HIP_TRY(c, strip_launch(c->prec, l, a, c->stream));
        } else {
            HIP_TRY(c, tb_steps(c->prec, c->A, c->B, c->flags, c->tb_lk, c->dsfrac, c->duin, c->tb_partials, pend, &nr, a, c->tb_t,
                                c->tb_k, kk, c->step, fi, nullptr, 0, c->stream));
        }
        pend += nr;
        c->nrec += nr;
        c->step += kk;
        left -= kk;
        std::swap(c->A, c->B);
        c->fields_fresh = false;
        c->replay_ok = false;
    }
    HIP_TRY(c, tb_force_flush(c->tb_partials, nparts, slots, c->hist, rec0, pend, step1, fi, c->stream));
    // records whose partials wait for one sum: of the two-step launches or of the one-step ones
    struct {
        bool pair = false;
        int n = 0, rec0 = 0;
        long step1 = 0;
    } wait;
    auto sum_waiting = [&]() {
        const int k = wait.n;
        wait.n = 0;
        return force_reduce(wait.pair ? c->pair.partials : c->partials, wait.pair ? c->pair.nslots : c->nslots, k, c->hist, wait.rec0,
                            wait.step1, fi, c->stream);
    };
    // the partials of the record of step `step`
    auto next_record = [&](bool pair, long step, double *&out) {
        const int nslots = pair ? c->pair.nslots : c->nslots;
        if (wait.n > 0 && (wait.pair != pair || wait.n == force_records(nslots))) {
            const hipError_t e = sum_waiting();
            if (e != hipSuccess) return e;
        }
        if (wait.n == 0) {
            wait.pair = pair;
            wait.rec0 = c->nrec;
            wait.step1 = step;
        }
        out = (pair ? c->pair.partials : c->partials) + 3 * (size_t)nslots * wait.n++;
        c->nrec++;
        return hipSuccess;
    };
    while (left > 0) {
        // two steps in one pass unless one of them records the force of a solid fraction (its moments
        // stay in registers), or the second a force that the pass does not sum (pair_plan); not under
        // per-kernel timing
        const bool second = records(c->step + 2);
        if (c->pair.on && !evs && left > 1 && !((second || records(c->step + 1)) && c->dsfrac) && !(second && !c->pair.seg)) {
            const PairOps ops = pair_ops(c->prec);
            if (records(c->step + 1)) {
                double *partials = nullptr;
                HIP_TRY(c, next_record(true, c->step + 1, partials));
                HIP_TRY(c, ops.force(c->pair, c->A, partials, a, c->stream));
            }
            double *sums = nullptr, *trip = nullptr;   // of the second step
            if (second) {
                HIP_TRY(c, next_record(true, c->step + 2, sums));
                trip = c->pair.fblk ? c->pair.trip : sums;
                if (c->pair.nnear == 0) trip = nullptr;
            }
            HIP_TRY(c, ops.step(c->pair, c->A, c->B, c->dsfrac, c->duin, c->macros, false, trip, a, c->stream));
            if (trip && c->pair.fblk) HIP_TRY(c, ops.block_sum(c->pair, sums, a, c->stream));
            c->step += 2;
            left -= 2;
            std::swap(c->A, c->B);
            c->fields_fresh = false;
            c->replay_ok = c->replay_pair = true;
            continue;
        }
        const int k = n - left;
        c->step++;
        left--;
        const bool force = records(c->step);
        StepBufs b = step_bufs(c, c->A, c->B);
        if (evs) {
            b.ev_bulk[0] = evs[2 * k];
            b.ev_bulk[1] = evs[2 * k + 1];
        }
        if (force) HIP_TRY(c, next_record(false, c->step, b.partials));
        HIP_TRY(c, plain_step(c->Q, c->prec, c->V, b, force, false, a, c->stream));
        std::swap(c->A, c->B);
        c->fields_fresh = false;
        c->replay_ok = true;
        c->replay_pair = false;
    }
    HIP_TRY(c, sum_waiting());
    return LBM_OK;
}

// The moments of the last step (and, in reference mode, the populations after its Update) are
// computed on request: the steps write only populations, and the last step is run again from
// its input buffer, which no later work has touched, with the moments on.  The populations it
// writes are those already in the output buffer, bit for bit (same kernel, same input), so the
// state does not change; the cost is one step, paid only when fields are read.
int ensure_fields(lbm_ctx *c) {
    if (c->fields_fresh) return LBM_OK;
    if (!c->replay_ok) return set_err(c, LBM_ERR_STATE, "fields of the current state are not available");
    if (ref_mode(c->cfg.bc_mode)) {
        if (c->rone.on)
            HIP_TRY(c, ref_one(c->rg, c->rone, c->rft, c->rf, c->rmac, c->rusr, c->rprof, c->rfpre, nullptr, 0, 0, c->stream));
        else HIP_TRY(c, ref_fused(c->rg, c->rft, c->rf, c->rmac, c->rusr, c->rprof, c->rfpre, c->stream));
    } else {
        const FusedArgs a = ctx_fused_args(c);
        if (c->replay_pair) HIP_TRY(c, pair_ops(c->prec).step(c->pair, c->B, c->A, c->dsfrac, c->duin, c->macros, true, nullptr, a, c->stream));
        else HIP_TRY(c, plain_step(c->Q, c->prec, c->V, step_bufs(c, c->B, c->A), false, true, a, c->stream));
    }
    c->fields_fresh = true;
    return LBM_OK;
}

extern "C" int lbm_step(lbm_ctx *c, int n) {
    if (!c) return LBM_ERR_INVALID;
    if (!c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_step before lbm_initialize");
    if (n < 0) return set_err(c, LBM_ERR_INVALID, "negative step count");
    if (n == 0) return LBM_OK;
    return step_n(c, n);
}

// ---- staged step (reference mode) ----
// The fused step leaves rf holding the next step's collided populations (the reference's first
// Collision acts on f = feq and changes nothing, and every later one is applied right after
// Update), so lbm_collide only opens the step; lbm_boundary, lbm_stream and lbm_update then run
// the reference's Streaming() in two parts and its Update() (followed by the next Collision, in
// place), leaving the same state as lbm_step(ctx, 1).
static int staged(lbm_ctx *c, int want, const char *name) {
    if (!c) return LBM_ERR_INVALID;
    if (!c->initialized) return set_err(c, LBM_ERR_STATE, std::string(name) + " before lbm_initialize");
    if (!ref_mode(c->cfg.bc_mode))
        return set_err(c, LBM_ERR_INVALID, std::string(name) + ": staged calls need a reference boundary mode "
                                                               "(the plain mode fuses the stages into one pass)");
    static const char *const order[4] = {"lbm_update (or nothing)", "lbm_collide", "lbm_boundary", "lbm_stream"};
    if (c->stage != want)
        return set_err(c, LBM_ERR_STATE, std::string(name) + " must follow " + order[want]);
    return LBM_OK;
}

extern "C" int lbm_collide(lbm_ctx *c) {
    int rc = staged(c, 0, "lbm_collide");
    if (rc != LBM_OK) return rc;
    // the staged fills write the ghost slots of both buffers, so the last fused step cannot be
    // rerun once the step is open: materialise its fields first
    rc = ensure_fields(c);
    if (rc != LBM_OK) return rc;
    c->replay_ok = false;
    rc = grow_hist(c, c->nrec + 2);
    if (rc != LBM_OK) return rc;
    c->step++;
    c->stage = 1;
    return LBM_OK;
}

extern "C" int lbm_boundary(lbm_ctx *c) {
    const int rc = staged(c, 1, "lbm_boundary");
    if (rc != LBM_OK) return rc;
    const int fi = c->cfg.force_interval;
    HIP_TRY(c, ref_fills(c->rg, c->rf, c->rft, c->stream));
    HIP_TRY(c, ref_boundary_pass(c, fi > 0 && c->step % fi == 0));
    c->stage = 2;
    return LBM_OK;
}

extern "C" int lbm_stream(lbm_ctx *c) {
    const int rc = staged(c, 2, "lbm_stream");
    if (rc != LBM_OK) return rc;
    HIP_TRY(c, ref_stream(c->rg, c->rf, c->rft, c->stream));
    std::swap(c->rf, c->rft);   // stream2: the ghost slots of both buffers are equal
    c->stage = 3;
    return LBM_OK;
}

extern "C" int lbm_update(lbm_ctx *c) {
    const int rc = staged(c, 3, "lbm_update");
    if (rc != LBM_OK) return rc;
    HIP_TRY(c, ref_update(c->rg, c->rf, c->rmac, c->rusr, c->rprof, c->rfpre, c->stream));
    c->stage = 0;
    c->fields_fresh = true;   // ref_update writes the moments and the populations after Update
    c->replay_ok = false;     // (it works in place: the fused kernel's input is gone)
    return LBM_OK;
}

extern "C" int lbm_step_timed(lbm_ctx *c, int n, double *ms) {
    if (!c || !ms) return LBM_ERR_INVALID;
    if (!c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_step_timed before lbm_initialize");
    hipEvent_t e0, e1;
    HIP_TRY(c, hipEventCreate(&e0));
    HIP_TRY(c, hipEventCreate(&e1));
    HIP_TRY(c, hipEventRecord(e0, c->stream));
    int rc = n > 0 ? step_n(c, n) : LBM_OK;
    HIP_TRY(c, hipEventRecord(e1, c->stream));
    HIP_TRY(c, hipEventSynchronize(e1));
    float t = 0.f;
    HIP_TRY(c, hipEventElapsedTime(&t, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms = t;
    return rc;
}

extern "C" int lbm_step_kernel_timed(lbm_ctx *c, int n, double *ms_steps, double *ms_bulk) {
    if (!c || !ms_steps || !ms_bulk) return LBM_ERR_INVALID;
    if (!c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_step_kernel_timed before lbm_initialize");
    if (c->cfg.bc_mode != LBM_BC_PLAIN) return set_err(c, LBM_ERR_INVALID, "lbm_step_kernel_timed times the plain mode");
    if (n <= 0 || n > 100000) return set_err(c, LBM_ERR_INVALID, "lbm_step_kernel_timed: n must be in [1, 100000]");
    std::vector<hipEvent_t> ev(2 * (size_t)n + 2, nullptr);
    auto release = [&]() {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
    };
    for (hipEvent_t &e : ev) {
        const hipError_t r = hipEventCreate(&e);
        if (r != hipSuccess) {
            e = nullptr;
            release();
            return set_err(c, LBM_ERR_HIP, std::string("hipEventCreate: ") + hipGetErrorString(r));
        }
    }
    hipError_t r = hipEventRecord(ev[2 * n], c->stream);
    int rc = r == hipSuccess ? step_n(c, n, ev.data()) : LBM_ERR_HIP;
    if (rc == LBM_OK) r = hipEventRecord(ev[2 * n + 1], c->stream);
    if (rc == LBM_OK && r == hipSuccess) r = hipEventSynchronize(ev[2 * n + 1]);
    float t = 0.f;
    double bulk = 0.0;
    if (rc == LBM_OK && r == hipSuccess) r = hipEventElapsedTime(&t, ev[2 * n], ev[2 * n + 1]);
    for (int k = 0; k < n && rc == LBM_OK && r == hipSuccess; k++) {
        float tk = 0.f;
        r = hipEventElapsedTime(&tk, ev[2 * k], ev[2 * k + 1]);
        bulk += tk;
    }
    release();
    if (rc != LBM_OK) return rc;
    if (r != hipSuccess) return set_err(c, LBM_ERR_HIP, std::string("lbm_step_kernel_timed: ") + hipGetErrorString(r));
    *ms_steps = t;
    *ms_bulk = bulk;
    return LBM_OK;
}

extern "C" int lbm_sync(lbm_ctx *c) {
    if (!c) return LBM_ERR_INVALID;
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    if (c->nrec > c->nrec_checked) {
        const int k = c->nrec - c->nrec_checked;
        HIP_TRY(c, output_forces(c));
        const double *const h = c->hist_copy.data() + 4 * (size_t)c->nrec_checked;
        const int first = c->nrec_checked;
        c->nrec_checked = c->nrec;
        for (int r = 0; r < k; r++)
            for (int d = 1; d < 4; d++) {
                const double v = h[4 * (size_t)r + d];
                if (!std::isfinite(v) || (c->cfg.force_limit > 0.0 && std::fabs(v) > c->cfg.force_limit))
                    return set_err(c, LBM_ERR_UNSTABLE, "force record " + std::to_string(first + r) + " (step " +
                                                          std::to_string((long)h[4 * (size_t)r]) + ") is not finite or exceeds force_limit");
            }
    }
    // the state itself, whether or not forces are recorded: the rest population of every live
    // node (a non-finite value reaches it within a step through the moments)
    if (c->initialized) {
        hipError_t e;
        if (ref_mode(c->cfg.bc_mode)) {
            const RefGeo &r = c->rg;
            const int gz = c->D == 3 ? r.g : 0;
            e = count_nonfinite(LBM_FP64, c->rf + r.g + r.rs * ((size_t)r.g + (size_t)r.ly * gz), r.rs, r.rs * r.ly, r.glx,
                                r.gly, r.glz, nullptr, 0, c->dbad, c->stream);
        } else {
            e = count_nonfinite(c->prec, c->A, c->geo.rs, c->geo.rs * c->geo.ny, c->geo.nx, c->geo.ny, c->geo.nz, c->flags,
                                c->geo.nxp, c->dbad, c->stream);
        }
        unsigned bad = 0;
        if (e == hipSuccess) e = hipMemcpyAsync(&bad, c->dbad, sizeof(unsigned), hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        if (e != hipSuccess) return set_err(c, LBM_ERR_HIP, std::string("lbm_sync: ") + hipGetErrorString(e));
        if (bad)
            return set_err(c, LBM_ERR_UNSTABLE, std::to_string(bad) + " nodes hold a non-finite rest population at step " +
                                                    std::to_string(c->step));
    }
    return LBM_OK;
}

extern "C" int lbm_set_step(lbm_ctx *c, long step) {
    if (!c) return LBM_ERR_INVALID;
    if (!c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_set_step before lbm_initialize");
    if (c->stage != 0) return set_err(c, LBM_ERR_STATE, "lbm_set_step inside a staged step");
    if (step < 0) return set_err(c, LBM_ERR_INVALID, "negative step");
    c->step = step;
    return LBM_OK;
}

// strip the ghost layers of a reference-mode plane (x fastest, interior only)
static void ref_strip(const lbm_ctx *c, const std::vector<double> &pad, double *out) {
    const RefGeo &r = c->rg;
    const int g = r.g, gz = c->D == 3 ? g : 0;
    size_t o = 0;
    for (int k = 0; k < r.glz; k++)
        for (int j = 0; j < r.gly; j++)
            for (int i = 0; i < r.glx; i++, o++)
                out[o] = pad[(size_t)(i + g) + (size_t)r.px * ((size_t)(j + g) + (size_t)r.ly * (k + gz))];
}

extern "C" int lbm_get_fields(lbm_ctx *c, double *p, double *u, double *v, double *w) {
    if (!c) return LBM_ERR_INVALID;
    if (!c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_get_fields before lbm_initialize");
    double *outs[4] = {p, u, v, w};
    if (c->stage == 0) {
        const int rc = ensure_fields(c);
        if (rc != LBM_OK) return rc;
    }
    HIP_TRY(c, output_fields(c, outs));
    return LBM_OK;
}

extern "C" int lbm_get_populations(lbm_ctx *c, double *f) {
    if (!c || !f) return set_err(c, LBM_ERR_INVALID, "null argument");
    if (!c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_get_populations before lbm_initialize");
    if (ref_mode(c->cfg.bc_mode)) {
        // between steps the reference's f is the state after Update; inside a staged step, the
        // state after the last stage
        if (c->stage == 0) {
            const int rc = ensure_fields(c);
            if (rc != LBM_OK) return rc;
        }
        const double *src = c->stage == 0 ? c->rfpre : c->rf;
        const RefGeo &r = c->rg;
        std::vector<double> pad(r.plane);   // one direction in the node layout
        for (int i = 0; i < c->Q; i++) {
            // rows of direction i: px elements every rs elements from element i*ds
            HIP_TRY(c, hipMemcpy2DAsync(pad.data(), sizeof(double) * r.px, src + (size_t)i * r.ds, sizeof(double) * r.rs,
                                        sizeof(double) * r.px, (size_t)r.ly * r.lz, hipMemcpyDeviceToHost, c->stream));
            HIP_TRY(c, hipStreamSynchronize(c->stream));
            ref_strip(c, pad, f + (size_t)i * c->N);
        }
        return LBM_OK;
    }
    const FusedArgs a = ctx_fused_args(c);
    double *tmp = nullptr;
    HIP_TRY(c, output_stage(c, &tmp));
    for (int i = 0; i < c->Q; i++) {
        HIP_TRY(c, plain_decode(c->Q, c->prec, c->A, tmp, c->flags, i, a, c->stream));
        HIP_TRY(c, output_staged(c, f + (size_t)i * c->N));
    }
    return LBM_OK;
}

extern "C" int lbm_set_populations(lbm_ctx *c, const double *f) {
    if (!c || !f) return set_err(c, LBM_ERR_INVALID, "null argument");
    if (!c->initialized) return set_err(c, LBM_ERR_STATE, "lbm_set_populations before lbm_initialize");
    if (ref_mode(c->cfg.bc_mode))
        return set_err(c, LBM_ERR_INVALID, "reference mode keeps ghost state; populations cannot be replaced");
    // the fields stay those of the last step (materialised now, while its input still exists)
    const int rc = ensure_fields(c);
    if (rc != LBM_OK) return rc;
    c->replay_ok = false;
    const FusedArgs a = ctx_fused_args(c);
    double *tmp = nullptr;
    HIP_TRY(c, hipMalloc(&tmp, sizeof(double) * c->N));
    for (int i = 0; i < c->Q; i++) {
        hipError_t e = hipMemcpyAsync(tmp, f + (size_t)i * c->N, sizeof(double) * c->N, hipMemcpyHostToDevice, c->stream);
        if (e == hipSuccess) e = plain_encode(c->Q, c->prec, c->A, tmp, c->flags, i, a, c->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        if (e != hipSuccess) {
            (void)hipFree(tmp);
            return set_err(c, LBM_ERR_HIP, std::string("lbm_set_populations: ") + hipGetErrorString(e));
        }
    }
    (void)hipFree(tmp);
    return LBM_OK;
}

extern "C" int lbm_get_forces(lbm_ctx *c, double *out, int max, int *count) {
    if (!c) return LBM_ERR_INVALID;
    HIP_TRY(c, output_forces(c));
    if (count) *count = c->nrec;
    const int n = std::min(max, c->nrec);
    if (out && n > 0) std::memcpy(out, c->hist_copy.data(), sizeof(double) * 4 * (size_t)n);
    return LBM_OK;
}

extern "C" int lbm_info_get(lbm_ctx *c, lbm_info *info) {
    if (!c || !info) return LBM_ERR_INVALID;
    std::memset(info, 0, sizeof(*info));
    info->lattice = c->Q;
    info->nx = c->geo.nx;
    info->ny = c->geo.ny;
    info->nz = c->geo.nz;
    info->pitch = c->cfg.bc_mode == LBM_BC_PLAIN ? c->geo.nxp : c->rg.px;
    info->nodes = c->N;
    const size_t esz = c->prec == LBM_FP64 ? 8 : c->prec == LBM_FP32 ? 4 : 2;
    info->state_bytes = c->cfg.bc_mode == LBM_BC_PLAIN ? esz * c->Q * c->geo.plane : 8 * c->Q * c->rg.plane;
    info->bytes_per_update = 2.0 * c->Q * (double)esz;
    info->step = c->step;
    info->solid_nodes = c->solid_nodes;
    info->boundary_nodes = c->near_nodes;
    info->nodes_per_lane = c->cfg.bc_mode == LBM_BC_PLAIN ? c->V : 1;
    return LBM_OK;
}
