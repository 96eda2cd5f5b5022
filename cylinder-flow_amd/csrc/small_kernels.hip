// small_kernels.hip -- host side of the several-steps-per-launch kernel (small_kernel.hpp): tiles, links,
// launches and the sum of its force records.
#include "small_kernel.hpp"

#include <algorithm>
#include <cstdlib>

namespace lbm {

// The force records of one launch: block r sums the ntiles partials of record r in a fixed order
// into hist[rec0 + r], whose step is step1 + r*fi.
__global__ void __launch_bounds__(256) k_tb_force(const double *__restrict__ partials, int ntiles,
                                                  double *__restrict__ hist, int rec0, long step1, int fi) {
    const int r = blockIdx.x;
    const double *P = partials + 3 * (size_t)r * ntiles;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    for (int j = threadIdx.x; j < ntiles; j += 256) {
        fx += P[3 * (size_t)j];
        fy += P[3 * (size_t)j + 1];
        fz += P[3 * (size_t)j + 2];
    }
    __shared__ double red[3 * 4];
    block_sum3<4>(fx, fy, fz, red);
    if (threadIdx.x == 0) {
        double *h = hist + 4 * (size_t)(rec0 + r);
        h[0] = (double)(step1 + (long)r * fi);
        h[1] = fx;
        h[2] = fy;
        h[3] = fz;
    }
}

// steps per launch: 7 (LBM_TB_DEPTH overrides, 1-10); FP64: with the 14 x 14 core of a 400 x 100
// domain's 28 x 28 tiles, 7 steps per launch measured fastest (2.54 us per step against 2.61 at
// 5 steps on 24 x 24 tiles and 2.60 at 8 on 30 x 30)
int tb_depth() {
    if (const char *e = std::getenv("LBM_TB_DEPTH")) {
        const int k = std::atoi(e);
        if (k >= 1 && k <= TB_KMAX) return k;
    }
    return 7;
}

size_t tb_lds_bytes(int prec, int T) { return tb_lds_size(T, prec == LBM_FP64 ? 8 : prec == LBM_FP32 ? 4 : 2); }

hipError_t tb_launch_f64(const TbLaunch &l, const FusedArgs &a, hipStream_t s);
hipError_t tb_launch_f32(const TbLaunch &l, const FusedArgs &a, hipStream_t s);
hipError_t tb_launch_f16(const TbLaunch &l, const FusedArgs &a, hipStream_t s);
hipError_t tb_launch_bf16(const TbLaunch &l, const FusedArgs &a, hipStream_t s);

int tb_tiles(const Geo &g, int T, int K, int *tiles_x) {
    const int W = T - 2 * K;
    *tiles_x = (g.nx + W - 1) / W;
    return *tiles_x * ((g.ny + W - 1) / W);
}

// the tile sides instantiated, and the tile side for a domain (leaving a core of at least 2 x 2
// nodes); LBM_TB_TILE overrides with any instantiated side that leaves a 2 x 2 core
static const int kTbSides[] = {24, 25, 26, 27, 28, 29, 30, 31, 32};

int tb_tile(const Geo &g, int K, int cus) {
    if (const char *e = std::getenv("LBM_TB_TILE")) {
        const int t = std::atoi(e);
        for (int T : kTbSides)
            if (t == T && t - 2 * K >= 2) return t;
    }
    // the side with the least (rounds of the CUs) x (positions per tile); measured best on
    // 400 x 100 (27), 600 x 150 (28), 800 x 200 (29) and 1000 x 250 (30) at 7 steps per launch
    int best = 32, tx = 0;
    long best_cost = -1;
    for (int T : kTbSides) {
        if (T - 2 * K < 2) continue;
        const long rounds = (tb_tiles(g, T, K, &tx) + cus - 1) / cus, cost = rounds * T * T;
        if (best_cost < 0 || cost < best_cost) {
            best = T;
            best_cost = cost;
        }
    }
    return best;
}

// record slots of the partials buffer: the force records of several launches are summed by one
// k_tb_force launch (a launch of its own costs about as much as a step)
int tb_records(int K) { return K > 128 ? K : 128; }

static hipError_t tb_launch(int prec, const TbLaunch &l, const FusedArgs &a, hipStream_t s) {
    switch (prec) {
    case LBM_FP64: return tb_launch_f64(l, a, s);
    case LBM_FP32: return tb_launch_f32(l, a, s);
    case LBM_FP16S: return tb_launch_f16(l, a, s);
    case LBM_BF16S: return tb_launch_bf16(l, a, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t tb_prepare(int prec, int T, const void *sfrac, const FusedArgs &a) {
    TbLaunch l{};
    l.T = T;
    l.sfrac = sfrac;
    l.prepare = true;
    hipError_t e = tb_launch(prec, l, a, nullptr);
    l.force = true;
    return e == hipSuccess ? tb_launch(prec, l, a, nullptr) : e;
}

// `steps` (<= K) steps from A into B, the first being step0 + 1; the partials of the force records
// among them go to record slots pend, pend + 1, ... (the caller keeps pend + steps within
// tb_records(K) and sums them with tb_force_flush).  Returns the number of records.
hipError_t tb_steps(int prec, const void *A, void *B, const uint8_t *flags, const uint16_t *lk, const void *sfrac,
                    const double *uin, double *partials, int pend, int *nrec, const FusedArgs &a, int T, int K, int steps,
                    long step0, int fi, void *keep, size_t keep_stride, hipStream_t s) {
    int tiles_x = 0;
    const int ntiles = tb_tiles(a.g, T, K, &tiles_x);
    const int nforce = fi > 0 ? (int)((step0 + steps) / fi - step0 / fi) : 0;
    *nrec = nforce;
    if (pend < 0 || pend + nforce > tb_records(K)) return hipErrorInvalidValue;
    if (T - 2 * K < 1 || K > TB_KMAX || steps < 1 || steps > K) return hipErrorInvalidValue;
    return tb_launch(prec, TbLaunch{A, B, flags, lk, sfrac, uin, partials, keep, keep_stride, T, K, steps, fi, tiles_x, ntiles, pend,
                                    step0, nforce > 0, false}, a, s);
}

hipError_t tb_force_flush(const double *partials, int nparts, int slots, double *hist, int rec0, int npend, long step1, int fi,
                          hipStream_t s) {
    if (npend <= 0) return hipSuccess;
    if (npend > slots || fi <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_tb_force, dim3(npend), dim3(256), 0, s, partials, nparts, hist, rec0, step1, fi);
    return hipGetLastError();
}

hipError_t strip_launch_f64(const StripLaunch &l, const FusedArgs &a, hipStream_t s);
hipError_t strip_launch_f32(const StripLaunch &l, const FusedArgs &a, hipStream_t s);
hipError_t strip_launch_f16(const StripLaunch &l, const FusedArgs &a, hipStream_t s);
hipError_t strip_launch_bf16(const StripLaunch &l, const FusedArgs &a, hipStream_t s);

hipError_t strip_launch(int prec, const StripLaunch &l, const FusedArgs &a, hipStream_t s) {
    switch (prec) {
    case LBM_FP64: return strip_launch_f64(l, a, s);
    case LBM_FP32: return strip_launch_f32(l, a, s);
    case LBM_FP16S: return strip_launch_f16(l, a, s);
    case LBM_BF16S: return strip_launch_bf16(l, a, s);
    default: return hipErrorInvalidValue;
    }
}

void strip_shape(const Geo &g, int prec, int cus, int steps, StripLaunch &l) {
    l.steps = steps;
    l.strips = (g.nx + 65 - 2 * steps) / (66 - 2 * steps);
    // a run per resident wave (2 per SIMD with FP64's registers, 4 otherwise), but no run shorter than
    // 4 rows: it would recompute more rows than it stores
    const int res = prec == LBM_FP64 ? 2 : 4, per_run = l.strips + (g.xper ? 0 : 1);
    const int runs = std::max(1, cus * 4 * res / per_run);
    l.rows = std::max((g.ny + runs - 1) / runs, 4);
    l.nwaves = per_run * ((g.ny + l.rows - 1) / l.rows);
}

}  // namespace lbm
