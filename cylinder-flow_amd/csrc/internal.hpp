// internal.hpp -- context and launcher interfaces shared by the kernel files and the
// C ABI (lbm_capi.cpp).  Not installed; include/lbm_capi.h is the public interface.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <thread>
#include <vector>

#include "lbm_capi.h"
#include "store.hpp"

namespace lbm {

// Device layout of the plain path.  Node arrays (flags, moments, solid fraction) are x fastest
// with rows padded to `nxp` (a multiple of 64 elements), so every wavefront row segment starts
// aligned:  node (x, y, z) = x + nxp*row,  row = y + ny*z,  plane = nxp*ny*nz.
// A population buffer holds, per row, the Q direction rows one after another (row-interleaved):
//   element (i, x, row) = i*ds + row*rs + x,   ds = nxp, rs = Q*nxp   (Q*plane elements)
// so one row's update reads and writes Q*nxp*sizeof(T) contiguous bytes (plus the source rows'
// stretches) instead of Q strips one plane apart.  ds = plane, rs = nxp gives the layout with
// one plane per direction, kept selectable (LBM_DIRECTION_PLANES) for comparison.
struct Geo {
    int nx, ny, nz, nxp;
    size_t plane;
    size_t ds, rs;
    int xper, yper, zper;
};

// population element of direction i at (x, row)
__host__ __device__ __forceinline__ size_t pel(const Geo &g, int i, uint32_t x, uint32_t row) {
    return (size_t)i * g.ds + (size_t)row * g.rs + x;
}

struct FusedArgs {
    Geo g;
    double tau;      // tau0 + 0.5 (FP64 path: f - (f - feq)/tau, the reference's form)
    double rtau;     // 1/tau rounded to nearest (for div_cr)
    float omega;     // 1/(tau0 + 0.5) (FP32 path)
    StoreParams sp;
};

// node flags
enum : uint8_t { FL_FLUID = 0, FL_SOLID = 1, FL_NEAR = 2 /* fluid with a solid neighbour */ };

// launch shape of every per-node kernel: blocks of `bx` threads along x, `gx` per row
struct Shape {
    int bx, gx;
};
Shape node_shape(const Geo &g);

// ---- initialisation of the node arrays (setup_kernels.hip) ----
struct SetupBody {
    int kind;   // lbm_config::body
    double cx, cy, cz, r2;
};
struct SetupFix {   // the rule of the FP32/16-bit fix list (init_plain); V nodes per lane
    int V;
    bool all, same_offsets;
};
// a node of the periodic x edges, or one whose lane reaches into the padding
__host__ __device__ inline bool fix_edge(const Geo &g, int V, int x) {
    return (g.xper && (x == 0 || x == g.nx - 1)) || (x == g.nx - 1 && g.nx % V != 0);
}
// a node of the inlet's or outlet's lane
__host__ __device__ inline bool fix_end_lane(const Geo &g, int V, int x) {
    const int x0 = x / V * V;
    return x0 == 0 || x0 + V >= g.nx;
}
// flags (padded layout) from the mask bytes (nx*ny*nz; null: from the body formula); sfrac: the caller's
// solid fraction on the device (nx*ny*nz) or null; counts: solid nodes, near nodes,
// nodes of the fix list
hipError_t setup_flags(int Q, uint8_t *flags, const uint8_t *mask, const double *sfrac, const SetupBody &b, const SetupFix &fix,
                       const Geo &g, unsigned *counts, hipStream_t s);
// per block of shape blk: 1 when it holds a node whose links or solid fraction carry force
hipError_t setup_forced(const uint8_t *flags, const double *sfrac, uint8_t *out, Shape blk, const Geo &g, hipStream_t s);
// per row: 1 when all its nodes are FL_FLUID, to both arrays
hipError_t setup_clean(const uint8_t *flags, uint8_t *clean, uint8_t *copy, const Geo &g, hipStream_t s);
// the solid fraction in the padded layout and the precision of the collision, 0 in the padding
hipError_t setup_sfrac(int prec, const double *in, void *out, const Geo &g, hipStream_t s);
// bounce-back links of the nodes for k_tb2d and k_strip: bit i-1 when direction i pulls from a solid node
// (after the outlet's clamp), bit 7+i when it pulls across a wall (not for the inlet's unknowns)
hipError_t setup_links9(const uint8_t *flags, uint16_t *lk, const Geo &g, hipStream_t s);

hipError_t plain_init(int Q, int prec, void *A, void *B, double *macros, const uint8_t *flags, const double *uin,
                      const double *xi, double perturb, uint64_t seed, const FusedArgs &a, hipStream_t s);
// launch shape of the fused kernels: V nodes per lane, at most 256 lanes per block
Shape lane_shape(const Geo &g, int V);
// launch shape of the FP64 kernel k_fused (and of its per-block force slots): 64-lane blocks on
// domains whose population buffer is at most 16 MB (the step is latency-bound there and wants
// every CU), otherwise lane_shape(g, 1)
Shape fp64_shape(const Geo &g, int Q);

// buffers of one fused step
struct StepBufs {
    const void *A;              // populations in (storage type)
    void *B;                    // populations out
    const uint8_t *flags;       // FL_* per node (padded layout)
    const uint32_t *fix;        // FP32/16-bit: nodes the packed path gets wrong (padded indices)
    const uint32_t *fixlk;      // their link words: bit i set when direction i pulls from a solid node
    int nfix;
    const int4 *rowwin;         // FP32/16-bit, per row (null: no mask links anywhere): the lanes
                                // [x, x + y) of the packed kernel hold mask links; their V nodes'
                                // link words start at element z of wlk
    const uint32_t *wlk;        // link words of the window nodes (0: no link, or a fix-list node)
    const uint32_t *link;       // the linked nodes the packed kernel handles (padded indices) ...
    const uint32_t *linklk;     // ... their link words
    const int *link_slot;       // ... and force partial slots (force steps: k_link_force)
    int nlink;
    const void *sfrac;          // solid fraction (FP64: double, else float) or null
    const double *uin;          // inlet velocity per (y, z)
    const int *block_slot;      // force partial slot per block (FP64) or per listed node (-1: none)
    double *partials;
    double *macros;             // p, u, v, w planes (written when macros_on)
    bool dense;                 // FP32/16-bit: one per-node pass over every node (k_dense_v)
                                // instead of the copies, the packed pass and the fix-up
    bool aligned_pull;          // 16-bit, two nodes per lane: aligned loads + lane shifts (k_fast_v)
    unsigned fast_lds;          // dynamic LDS bytes per k_fast_v block (caps its blocks per CU; 0: none)
    hipEvent_t ev_bulk[2];      // when set: recorded just before and after the step's bulk kernel
                                // (k_fast_v, k_dense_v, or k_fused in FP64), on the step's stream
};
hipError_t plain_step(int Q, int prec, int V, const StepBufs &b, bool force, bool macros_on, const FusedArgs &a,
                      hipStream_t s);
hipError_t fast_step_f32(int Q, int V, const StepBufs &b, bool force, bool mac, const FusedArgs &a, hipStream_t s);
hipError_t fast_step_f16(int Q, int V, const StepBufs &b, bool force, bool mac, const FusedArgs &a, hipStream_t s);
hipError_t fast_step_bf16(int Q, int V, const StepBufs &b, bool force, bool mac, const FusedArgs &a, hipStream_t s);
// two D3Q27 steps per pass over memory (pair_kernel.hpp): WX x WY columns over runs of cz planes.
// The words and lists are built once from the mask (pair_plan).
struct PairSeg {   // the nodes next to the mask among 64 along a row: how many come before them, and which
    uint32_t base, lo, hi, unused;
};
struct PairPlan {
    bool on = false;
    int tiles_x = 0, tiles_y = 0, cz = 0, chunks = 0;
    uint32_t *bw = nullptr;       // per node (padded layout): bit i set when direction i bounces back
    uint32_t *tflag = nullptr;    // per column, (nz + 31) / 32 words: bit k set when plane k of the column
                                  // and its rim holds a non-zero bw
    // Force partials in the slots of the one-step path of the domain, so that the sums are the same:
    // one per node next to the mask (nlink of them, node order) ...
    uint32_t *link = nullptr;     // the nodes ...
    uint32_t *linklk = nullptr;   // ... their mask links (bit i: direction i pulls from a solid node) ...
    int *link_slot = nullptr;     // ... and slots (0, 1, ...)
    int nlink = 0;
    // ... or one per block of fbx nodes of a row (fgx per row) that holds such a node
    uint32_t *fblk = nullptr;     // the blocks in slot order (null: per node)
    int fbx = 0, fgx = 0;
    int nslots = 0;
    double *partials = nullptr;   // force_bytes(nslots)
    // force of the second step of a pair: the nodes next to the mask (nnear of them) by segment, and with
    // per-block slots their three sums (else those are the slots)
    PairSeg *seg = nullptr;
    int nnear = 0;
    double *trip = nullptr;
};
struct PairOps {   // a storage format's column, LDS bytes and launchers
    int wx, wy;
    size_t lds;
    hipError_t (*prepare)();
    hipError_t (*step)(const PairPlan &p, const void *A, void *B, const void *sfrac, const double *uin, double *macros,
                       bool mac, double *trip, const FusedArgs &a, hipStream_t s);   // trip: see PairPlan (null: no force)
    hipError_t (*force)(const PairPlan &p, const void *A, double *partials, const FusedArgs &a, hipStream_t s);
    hipError_t (*block_sum)(const PairPlan &p, double *partials, const FusedArgs &a, hipStream_t s);
};
PairOps pair_ops(int prec);
// the plan of a domain; p.on stays false where the two-step kernel does not apply (pair.cpp).
// flags: on the device, complete on stream s; packed: the one-step path is k_fast_v alone; near_nodes: the nodes next to the mask, in node order;
// block_slot: the one-step path's slot per block of shape `blk` (empty: its slots are per node)
hipError_t pair_plan(PairPlan &p, int prec, const Geo &g, const uint8_t *flags, bool same_offsets, bool packed,
                     const std::vector<uint32_t> &near_nodes, const std::vector<int> &block_slot, Shape blk, hipStream_t s);
// fills p.bw, p.tflag and p.linklk (pair_words.hip)
// masks: per 64 nodes along a row, those next to the mask
hipError_t pair_words(const PairPlan &p, const PairOps &ops, const uint8_t *flags, unsigned long long *masks, const Geo &g,
                      hipStream_t s);
void pair_free(PairPlan &p);
// several D2Q9 steps per launch (small_kernel.hpp): K steps at most, T x T tiles
// (tb_choose), tb_tiles(g, T, K) blocks with tb_lds_bytes(prec, T) of LDS each
size_t tb_lds_bytes(int prec, int T);
int tb_tiles(const Geo &g, int T, int K, int *tiles_x);
// steps per launch and tile side of a domain with the force every fi steps (0: never)
void tb_choose(const Geo &g, int prec, int fi, int cus, int &K, int &T);
// before the first launch: the LDS limit of the kernels for side T (sfrac: null or not) on this device
hipError_t tb_prepare(int prec, int T, const void *sfrac, const FusedArgs &a);
// tb_steps: `steps` (<= K) steps in one launch; the partials of its force records go to record
// slots pend, pend + 1, ... of `partials` (tb_records() slots of ntiles * 3 doubles); *nrec = their
// count.  keep (null: none): the state after step k < steps of the launch goes to keep + (k - 1) * keep_stride (elements)
int tb_records(int K);
hipError_t tb_steps(int prec, const void *A, void *B, const uint8_t *flags, const uint16_t *lk, const void *sfrac,
                    const double *uin, double *partials, int pend, int *nrec, const FusedArgs &a, int T, int K, int steps,
                    long step0, int fi, void *keep, size_t keep_stride, hipStream_t s);
// sums npend record slots (of `slots`) of nparts triples each into hist[rec0 ...], the first at step step1
hipError_t tb_force_flush(const double *partials, int nparts, int slots, double *hist, int rec0, int npend, long step1, int fi,
                          hipStream_t s);
// several D2Q9 steps per pass over memory on large domains (strip_kernel.hpp): `steps` (2..4) steps
// from A into B by nwaves waves, strips (66 - 2 steps columns each) x runs of `rows` rows; bit l of rec:
// step l + 1 records the force, its partials go to record slot pend, pend + 1, ... (nwaves triples each)
struct StripLaunch {
    const void *A;
    void *B;
    const uint16_t *lk;   // setup_links9
    const void *sfrac;
    const double *uin;
    double *partials;
    int steps, strips, rows, nwaves, pend;
    uint32_t rec;
};
constexpr int STRIP_K = 4;   // steps per pass
hipError_t strip_launch(int prec, const StripLaunch &l, const FusedArgs &a, hipStream_t s);
// fills steps, strips, rows and nwaves
void strip_shape(const Geo &g, int prec, int cus, int steps, StripLaunch &l);

// force partials: a buffer of force_bytes(nslots) keeps those of force_records(nslots) steps, 3 * nslots
// doubles each; force_reduce sums the first nrec of them into hist[rec], hist[rec + 1], ... (steps step,
// step + every, ...)
int force_records(int nslots);
size_t force_bytes(int nslots);
hipError_t force_reduce(double *partials, int nslots, int nrec, double *hist, int rec, long step, int every, hipStream_t s);
// FP64 <-> storage conversion of one direction's populations (physical nodes, x fastest)
hipError_t plain_decode(int Q, int prec, const void *A, double *out, const uint8_t *flags, int dir,
                        const FusedArgs &a, hipStream_t s);
hipError_t plain_encode(int Q, int prec, void *A, const double *in, const uint8_t *flags, int dir,
                        const FusedArgs &a, hipStream_t s);
// number of non-finite values of one direction over a box of nodes (see k_count_nonfinite) into
// *bad (device memory), for storage format prec
hipError_t count_nonfinite(int prec, const void *base, size_t sy, size_t sz, int nx, int ny, int nz,
                           const uint8_t *flags, int fpitch, unsigned *bad, hipStream_t s);
// moment plane k (p, u, v, w) at the physical nodes; 0 at solid nodes
hipError_t macros_extract(const double *macros, const uint8_t *flags, double *out, int k, const Geo &g, hipStream_t s);

// the moment planes of mask (bit k: p, u, v, w) one after another, physical nodes, 0 at solid nodes
hipError_t plain_fields(const double *macros, const uint8_t *flags, double *out, unsigned mask, const Geo &g, hipStream_t s);

// ---- reference mode (FP64, ghost-padded SoA) ----
struct RefGeo {
    int Q, D, g;                 // ghost width 3 (3D) / 2 (2D)
    int glx, gly, glz;           // interior extents
    int lx, ly, lz;              // padded extents
    int px;                      // row pitch in elements (>= lx; 3D rows start 256-byte aligned)
    size_t plane;                // px*ly*lz
    size_t ds, rs;               // population element (ii, i, j, k) = ii*ds + i + rs*(j + ly*k)
    double tau0, u0;
    int variant;                 // D2Q9: 0 the MPI variant, 1 the single-node variant
    unsigned lds;                // dynamic LDS per block of the fused kernel (caps its blocks per CU; 0: none)
};
hipError_t ref_init(const RefGeo &r, double *f, double *ft, double *mac, uint8_t *usr, const int32_t *ran,
                    int body, double cx, double cy, double cz, double r2, uint64_t seed, hipStream_t s);
hipError_t ref_fills(const RefGeo &r, double *f, double *ft, hipStream_t s);
// list (may be null: sweep the interior): the nodes usrbc can change, nlist of them
hipError_t ref_usrbc(const RefGeo &r, double *f, const uint8_t *usr, const uint32_t *list, int nlist, hipStream_t s);
// with_usrbc: the same pass also applies usrbc (in place of a separate ref_usrbc before it)
hipError_t ref_mem(const RefGeo &r, double *f, const uint8_t *usr, double *partials, int nblk,
                   double *hist, int rec, long step, bool with_usrbc, hipStream_t s);
// fpre (may be null): receives the pulled populations, i.e. the reference's f after Update
hipError_t ref_fused(const RefGeo &r, const double *f, double *ft, double *mac, const uint8_t *usr,
                     const double *prof, double *fpre, hipStream_t s);
// the staged step's pull (ft = stream1 of f at the interior nodes) and its Update + next
// Collision in place on f (fpre as for ref_fused)
hipError_t ref_stream(const RefGeo &r, const double *f, double *ft, hipStream_t s);
hipError_t ref_update(const RefGeo &r, double *f, double *mac, const uint8_t *usr, const double *prof, double *fpre,
                      hipStream_t s);
int ref_mem_blocks(const RefGeo &r);
// One 2D step in one launch: every pulled value straight from where the fills and usrbc would have copied
// it from (ref_resolve), so neither buffer's ghosts are touched.
struct RefLink {       // a momentum-exchange link: f_i at the fluid node + f_opp at the solid one
    int a, b, b0;      // elements of f: the first, the second after usrbc, the second's origin before the fills
    int dir;
};
struct RefOne {
    bool on = false;
    int *special = nullptr;     // per node: row of `rows`, -1 where every source is the plain neighbour
    int *rows = nullptr;        // 9 source elements of each special node
    RefLink *links = nullptr;   // in node order, directions in order
    int nlinks = 0;
};
// false: some source is a ghost slot that no fill of the same step writes (the values of an earlier
// step then stay in the ghosts, which only the separate fills keep)
bool ref_resolve(const RefGeo &r, const std::vector<uint8_t> &usr, std::vector<int> &special, std::vector<int> &rows,
                 std::vector<RefLink> &links);
// hist non-null: the force record of the step (from the same input) goes to hist[4 * rec ...]
hipError_t ref_one(const RefGeo &r, const RefOne &o, const double *f, double *ft, double *mac, const uint8_t *usr,
                   const double *prof, double *fpre, double *hist, int rec, long step, hipStream_t s);
// the same sum after the separate fills and usrbc
hipError_t ref_one_force(const RefGeo &r, const RefOne &o, const double *f, double *hist, int rec, long step, hipStream_t s);
// the interior (ghost layers stripped) of the moment planes of mask, one after another
hipError_t ref_fields(const RefGeo &r, const double *mac, double *out, unsigned mask, hipStream_t s);

// ---- adjoint (plain mode) ----
struct AdjArgs {
    FusedArgs f;
    double alpha;        // window weight of this step (dJ/dFx)
    double alpha_next;   // window weight of the next step
};
// rowclean: per row (ny*nz bytes), 1 when no node of the row is solid or next to a solid node;
// all_fast: every row is clean and none lies on a periodic y/z edge (the straight-line kernel alone)
hipError_t adj_step(int Q, int prec, const void *H, const void *mu_next, void *mu, const uint8_t *flags,
                    const void *sfrac, const double *uin, void *dJds, double *dJdu_rows, const uint8_t *rowclean,
                    bool all_fast, const AdjArgs &a, hipStream_t s);
// weight of step m: w within n0 .. n1, else 0
struct AdjWindow {
    int n0, n1;
    double w;
    __host__ __device__ double at(int m) const { return m >= n0 && m <= n1 ? w : 0.0; }
};
// several reverse steps per launch on small non-periodic D2Q9 domains (adjoint_small.hip): steps m, m - 1, ...
// (steps <= K of them) from mun = mu_{m+1} to mu; H: H_{m-1}, the states before it `stride` elements apart
// below it, but for the last of the launch, which is Hlast; tiles as tb_steps
struct AdjSmall {
    const void *H, *Hlast;
    size_t stride;
    const void *mun;
    void *mu;
    const uint8_t *flags;
    const uint16_t *lk;
    const void *sfrac;
    const double *uin;
    double *dJds, *dJdu;
    AdjWindow win;
    int m, T, K, steps;
    bool prepare;   // only set the kernel's LDS limit on the current device
};
hipError_t adj_small(int prec, const AdjSmall &l, const FusedArgs &a, hipStream_t s);
hipError_t adj_init(int Q, int prec, const void *mu1, const uint8_t *flags, const double *uin,
                    const double *xi, double perturb, uint64_t seed, double alpha1, double *dJdu_rows,
                    const FusedArgs &a, hipStream_t s);
hipError_t adj_reduce_ds(int prec, const void *dJds, double *out, const Geo &g, hipStream_t s);

}  // namespace lbm

struct SnapshotJob;

struct lbm_ctx {
    lbm_config cfg{};
    int Q = 0, D = 0, prec = 0;
    lbm::Geo geo{};
    size_t N = 0;           // physical nodes
    hipStream_t stream = nullptr;
    std::string err;

    // host-side set-up inputs
    std::vector<uint8_t> solid;     // N
    std::vector<double> sfrac;      // N or empty
    std::vector<double> uin;        // ny*nz
    std::vector<double> xi;         // N or empty (injected perturbation)
    std::vector<int32_t> ran;       // padded box or empty (reference mode)
    bool uin_set = false;
    int solid_nodes = 0, near_nodes = 0;

    // plain-mode device state
    void *A = nullptr, *B = nullptr;
    uint8_t *flags = nullptr;
    uint8_t *rowclean = nullptr;    // per row: 1 when every node is fluid with no solid neighbour
    bool adj_all_fast = false;      // every row clean and off the periodic y/z edges
    void *dsfrac = nullptr;
    double *duin = nullptr;
    double *macros = nullptr;       // 4 planes of FP64
    int *block_slot = nullptr;
    double *partials = nullptr;
    int nslots = 0;
    int tb_k = 0;                   // D2Q9 small domains: steps per temporally blocked launch (0: off)
    int tb_t = 0;                   // and its tile side
    bool strip = false;             // D2Q9 large domains: STRIP_K steps per pass (strip_kernel.hpp)
    int cus = 0;                    // compute units of the device
    double *tb_partials = nullptr;  // force partials per tile or wave (tb_records(...) record slots)
    uint16_t *tb_lk = nullptr;      // and each node's bounce-back links (setup_links9)
    uint32_t *fix = nullptr;        // FP32/16-bit: nodes recomputed per node after the packed path
    uint32_t *fixlk = nullptr;      // their link words
    int nfix = 0;
    int4 *rowwin = nullptr;         // FP32/16-bit: per-row windows of mask links (see StepBufs)
    uint32_t *wlk = nullptr;
    uint32_t *link = nullptr;       // mask-neighbour nodes handled by the packed kernel, their link
    uint32_t *linklk = nullptr;     // words and force slots (for k_link_force)
    int *link_slot = nullptr;
    int nlink = 0;
    lbm::PairPlan pair;             // D3Q27: two steps per pass
    int V = 1;                      // nodes per lane of the fused kernel
    bool aligned_pull = true;
    bool dense = false;             // FP32/16-bit: per-node pass over every node (see StepBufs)
    unsigned fast_lds = 0;

    unsigned *dbad = nullptr;       // lbm_sync's count of non-finite populations (device)
    double *noalloc_scratch = nullptr;   // lbm_get_fields_noalloc's staging array on this device
    std::string noalloc_err;

    // force history (device + host copy)
    double *hist = nullptr;
    int hist_cap = 0, nrec = 0, nrec_checked = 0;

    // reference-mode device state
    lbm::RefGeo rg{};
    double *rf = nullptr, *rft = nullptr, *rmac = nullptr, *rprof = nullptr, *rfpre = nullptr;
    uint8_t *rusr = nullptr;
    lbm::RefOne rone;               // 2D: one launch per step
    uint32_t *rsurf = nullptr;      // interior solid nodes with a fluid neighbour (usrbc's work list)
    int nsurf = 0;

    bool initialized = false;
    long step = 0;
    // Fields (and, in reference mode, the populations after Update) are written on request, not
    // every step: fields_fresh says they belong to the current state; otherwise replay_ok says the
    // last step's input buffer is intact, so rerunning that step with the moments on rewrites the
    // same populations and fills them in (replay_pair: that pass was two steps).
    bool fields_fresh = true;
    bool replay_ok = false;
    bool replay_pair = false;
    // results on their way to the caller (output.cpp): device buffer and pinned memory, kept for reuse,
    // and the force records already on the host
    double *out_dev = nullptr, *out_pin = nullptr;
    size_t out_elems = 0, out_pinned = 0;
    std::vector<double> hist_copy;
    // snapshot staging: device buffer (plain mode) and pinned host buffer, kept for reuse
    double *snap_dev = nullptr, *snap_host = nullptr;
    size_t snap_elems = 0;
    // staged step (reference mode): 0 between steps (rf holds the next step's collided
    // populations, rfpre the populations after Update), 1 after lbm_collide, 2 after
    // lbm_boundary, 3 after lbm_stream
    int stage = 0;

    SnapshotJob *snap = nullptr;
};

// materialise the fields of the last step (see lbm_capi.cpp); LBM_OK or an LBM_ERR_* code
int ensure_fields(lbm_ctx *c);
// device results into the caller's arrays (output.cpp)
hipError_t output_fields(lbm_ctx *c, double *const *outs);
hipError_t output_stage(lbm_ctx *c, double **dev);
hipError_t output_staged(lbm_ctx *c, double *dst);
hipError_t output_forces(lbm_ctx *c);
void output_free(lbm_ctx *c);
// the address of lbm_get_fields_noalloc's staging array on the current device (noalloc.hip)
int noalloc_setup(double **out, std::string &err);
