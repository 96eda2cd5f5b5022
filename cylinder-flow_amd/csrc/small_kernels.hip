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

// Steps per launch and tile side of a domain: the least microseconds per step by a model of a launch of K
// steps over T x T tiles, in rounds of one tile per CU (FP64, whose tile fills the LDS) or two:
//   t0 + rounds of the CUs * a K + tiles per CU * b * wave-steps of the busiest SIMD (+ c T^2 per round, FP64),
// a and b larger by a1, b1 in a step that records the force.  The constants are a least-squares fit to 126
// launches per format from 48x32 to 1000x250, 4 to 10 steps, the force every step and every 10 (FP64: 2 % rms,
// FP32 and 16 bits: 9 %).  More steps save launches, until the halo makes the tiles too many for the CUs: us
// per step with the force every 10 steps, always 7 steps per launch / this choice:
//              FP64           FP32           FP16
//   48x32      1.78 / 1.51    1.28 / 1.06    1.41 / 1.13
//   400x100    2.03 / 1.93    1.38 / 1.31    1.51 / 1.40
//   512x128    2.38 / 2.25    1.55 / 1.48    1.68 / 1.58
//   600x150    3.78 / 2.54    1.89 / 1.65    2.03 / 1.73
//   800x200    5.68 / 4.02    2.80 / 2.66    2.99 / 2.73
//   1000x250   8.05 / 6.22    4.97 / 3.67    5.53 / 3.99
// (with the force every step 10.7 / 7.51, 8.20 / 4.70 and 8.35 / 4.67 on the last; a few percent of each is
// the kept states' test, which launches with force records no longer hold).  t0 lies 0.3 (FP64) below and 0.8
// above the fit's, where the least measured launches of 400x100 and 512x128 are taken.
// LBM_TB_DEPTH (1-10) fixes the steps, LBM_TB_TILE the side (one that is instantiated and leaves a 2 x 2 core).
static const int kTbSides[] = {24, 25, 26, 27, 28, 29, 30, 31, 32};

void tb_choose(const Geo &g, int prec, int fi, int cus, int &K, int &T) {
    const bool f64 = prec == LBM_FP64;
    const double phi = fi > 0 ? 1.0 / fi : 0.0;
    const double t0 = f64 ? 2.2 : 3.2, a = f64 ? 0.606 + 0.288 * phi : 0.494 + 0.08 * phi,
                 b = f64 ? 0.287 + 0.185 * phi : 0.304 + 0.32 * phi, c = f64 ? 0.0042 : 0.0;
    int only_k = 0, only_t = 0;
    if (const char *e = std::getenv("LBM_TB_DEPTH")) only_k = std::atoi(e);
    if (only_k < 1 || only_k > TB_KMAX) only_k = 0;
    if (const char *e = std::getenv("LBM_TB_TILE"))
        for (int side : kTbSides)
            if (std::atoi(e) == side && (only_k ? side - 2 * only_k : side - 4) >= 2) only_t = side;
    double best = -1.0;
    K = T = 0;
    for (int k = only_k ? only_k : 2; k <= (only_k ? only_k : TB_KMAX); k++)
        for (int side : kTbSides) {
            const int W = side - 2 * k;
            if (W < 2 || (only_t && side != only_t)) continue;
            int tx = 0, waves = 0;
            const int n = tb_tiles(g, side, k, &tx), per_cu = (n + cus - 1) / cus, at_once = f64 ? 1 : 2;
            for (int m = 0; m < k; m++) waves += ((W + 2 * m) * (W + 2 * m) + 255) / 256;
            const double t = (t0 + (per_cu + at_once - 1) / at_once * a * k + per_cu * (b * waves + c * side * side)) / k;
            if (best < 0.0 || t < best) {
                best = t;
                K = k;
                T = side;
            }
        }
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
    if (T - 2 * K < 1 || K > TB_KMAX || steps < 1 || steps > K || (keep && nforce > 0)) return hipErrorInvalidValue;
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
