// adjoint.cpp -- checkpointed discrete-adjoint driver (lbm_adjoint; no reference counterpart).
//
// Forward: steps 1..n1 from the initial state, drag recorded every step, the state saved
// every K steps (checkpoints H_0, H_K, ...).  Reverse: for each segment, newest first, the
// checkpoint is restored and the segment's states H_{m0} .. H_{m0+n-1} are recomputed into
// a device-resident store (up to K states: with 288 GB of HBM a whole segment of a 1.8 M-node
// D3Q27 FP32 run, ~48 GB at K = 250, stays on the GPU), then one reverse kernel per step
// turns mu_{m+1} into mu_m.  Cost: the recompute is one forward pass; each reverse step
// moves 3Q values per node against the forward's 2Q.
#include <cmath>
#include <cstring>

#include "internal.hpp"

using namespace lbm;

static int aerr(lbm_ctx *c, int code, const std::string &m) {
    c->err = m;
    return code;
}

#define ATRY(expr)                                                                                     \
    do {                                                                                               \
        hipError_t e__ = (expr);                                                                       \
        if (e__ != hipSuccess) {                                                                       \
            rc = aerr(c, LBM_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e__));             \
            goto done;                                                                                 \
        }                                                                                              \
    } while (0)

FusedArgs ctx_fused_args(const lbm_ctx *c);
StepBufs step_bufs(const lbm_ctx *c, const void *A, void *B);

extern "C" int lbm_adjoint(lbm_ctx *c, int n0, int n1, double scale, int K, double *J, double *dJ_ds,
                           double *dJ_duin, double *ms_forward, double *ms_adjoint) {
    if (!c) return LBM_ERR_INVALID;
    if (c->cfg.bc_mode != LBM_BC_PLAIN) return aerr(c, LBM_ERR_INVALID, "the adjoint covers the plain boundary mode");
    if (c->prec != LBM_FP64 && c->prec != LBM_FP32) return aerr(c, LBM_ERR_INVALID, "the adjoint needs FP64 or FP32 storage");
    if (!c->initialized || c->step != 0) return aerr(c, LBM_ERR_STATE, "lbm_adjoint needs a freshly initialised context (step 0)");
    if (n0 < 1 || n1 < n0) return aerr(c, LBM_ERR_INVALID, "need 1 <= n0 <= n1");
    if (K <= 0 || K > n1) K = n1;
    const int K_asked = K;
    const Geo &g = c->geo;
    const int Q = c->Q;
    const size_t esz = c->prec == LBM_FP64 ? 8 : 4;
    const size_t SZ = esz * Q * g.plane;
    // Freed device memory is cleared before it is given out again, at about 40 GB/s behind the program's
    // back: a program that evaluates gradients one after another runs into that once it has gone through
    // the card's memory, and then pays for every byte of the store (192x96x96 FP32, 400 steps, K = 50, 11.4 GB
    // per evaluation: 295 ms on average over 80 evaluations, 115 for each of the first 24; 209 ms with the split
    // below; 96x48x48 FP64, 300 steps, 200 evaluations, K = 7 / 20 / 50: 101 / 74 / 110 ms on average, 47 / 70 /
    // 68 with it).  From 1 GB on the segments are therefore of sqrt(n1) steps where that makes fewer states, at the
    // same recompute; the copies of the added checkpoints take 1-3 %.  Below, and up to 4 GB where several steps
    // go into a launch and short segments leave more remainders, the segments are those asked for.
    {
        const int root = (int)std::ceil(std::sqrt((double)n1)), states = (n1 + K - 1) / K + K;
        if ((double)SZ * states >= (c->tb_k >= 2 ? 4e9 : 1e9) && (n1 + root - 1) / root + root < states) K = root;
    }
    const int nseg = (n1 + K - 1) / K;
    int rc = LBM_OK;
    void *ckpt = nullptr, *store = nullptr, *mu0 = nullptr, *mu1 = nullptr;
    double *dJds = nullptr, *dJdu = nullptr, *tmp = nullptr, *dxi = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr, e2 = nullptr;
    float tf = 0.f, ta = 0.f;
    const FusedArgs fa = ctx_fused_args(c);
    const AdjWindow win{n0, n1, scale / (double)(n1 - n0 + 1)};
    const int fi_saved = c->cfg.force_interval;
    std::vector<double> hist;
    size_t freeb = 0, totalb = 0;

    output_free(c);   // the kept output buffer's memory counts as free here
    (void)hipMemGetInfo(&freeb, &totalb);
    // (the store of the segments asked for: what was refused does not depend on the split above)
    const int asked = (n1 + K_asked - 1) / K_asked + K_asked + 2;
    if ((double)SZ * asked + 8.0 * g.plane * 2 > 0.95 * (double)freeb)
        return aerr(c, LBM_ERR_NOMEM, "adjoint store (" + std::to_string((double)SZ * asked / 1e9) +
                                         " GB) exceeds free device memory; lower checkpoint_every");
    ATRY(hipMalloc(&ckpt, SZ * nseg));
    if (K > 1) ATRY(hipMalloc(&store, SZ * (K - 1)));   // a segment's states but its first, which is the checkpoint
    ATRY(hipMalloc(&mu0, SZ));
    ATRY(hipMalloc(&mu1, SZ));
    ATRY(hipMalloc(&dJds, sizeof(double) * g.plane));
    ATRY(hipMalloc(&dJdu, sizeof(double) * g.ny * g.nz));
    ATRY(hipMemsetAsync(mu0, 0, SZ, c->stream));
    ATRY(hipMemsetAsync(mu1, 0, SZ, c->stream));
    ATRY(hipMemsetAsync(dJds, 0, sizeof(double) * g.plane, c->stream));
    ATRY(hipMemsetAsync(dJdu, 0, sizeof(double) * g.ny * g.nz, c->stream));
    if (!c->xi.empty()) {
        ATRY(hipMalloc(&dxi, sizeof(double) * c->N));
        ATRY(hipMemcpyAsync(dxi, c->xi.data(), sizeof(double) * c->N, hipMemcpyHostToDevice, c->stream));
    }
    ATRY(hipEventCreate(&e0));
    ATRY(hipEventCreate(&e1));
    ATRY(hipEventCreate(&e2));

    if (c->tb_k >= 2) {
        AdjSmall l{};
        l.sfrac = c->dsfrac;
        l.T = c->tb_t;
        l.K = c->tb_k;
        l.steps = 1;
        l.prepare = true;
        ATRY(adj_small(c->prec, l, fa, c->stream));
    }

    // ---- forward with checkpoints, drag every step ----
    c->cfg.force_interval = 1;
    ATRY(hipEventRecord(e0, c->stream));
    for (int k = 0; k < nseg; k++) {
        ATRY(hipMemcpyAsync((char *)ckpt + SZ * k, c->A, SZ, hipMemcpyDeviceToDevice, c->stream));
        const int n = (k + 1) * K <= n1 ? K : n1 - k * K;
        rc = lbm_step(c, n);
        if (rc != LBM_OK) goto done;
    }
    ATRY(hipEventRecord(e1, c->stream));

    // ---- reverse sweep ----
    {
        void *mun = mu0, *mu = mu1;   // mun holds mu_{m+1} (zero beyond n1)
        for (int k = nseg - 1; k >= 0; k--) {
            const int m0 = k * K;
            const int n = (m0 + K <= n1) ? K : n1 - m0;
            auto state = [&](int t) { return t == 0 ? (char *)ckpt + SZ * k : (char *)store + SZ * (t - 1); };
            for (int t = 0; t + 1 < n;) {
                char *const H = state(t), *const next = state(t + 1);
                // Small D2Q9 domains: tb_k steps per launch, every state stored (400x100 FP64: 1000 steps'
                // recompute 3.8 -> 2.0 ms).  D3Q27 stays at one step per launch: the write of every state
                // bounds it either way (192x96x96 FP32, two steps per pass with both states stored, 75 us
                // per step against 67: the read a second step saves came from the last-level cache).
                if (c->tb_k >= 2 && n - 1 - t >= 2) {
                    int nrec = 0;
                    const int steps = n - 1 - t < c->tb_k ? n - 1 - t : c->tb_k;
                    ATRY(tb_steps(c->prec, H, next + SZ * (steps - 1), c->flags, c->tb_lk, c->dsfrac, c->duin, c->tb_partials, 0, &nrec, fa,
                                  c->tb_t, c->tb_k, steps, m0 + t, 0, next, SZ / esz, c->stream));
                    t += steps;
                } else {
                    ATRY(plain_step(Q, c->prec, c->V, step_bufs(c, H, next), false, false, fa, c->stream));
                    t++;
                }
            }
            for (int t = n - 1; t >= 0;) {
                const int m = m0 + t + 1;
                if (c->tb_k >= 2 && t >= 1) {   // the steps m, m - 1, ... of a launch
                    const int steps = t + 1 < c->tb_k ? t + 1 : c->tb_k;
                    ATRY(adj_small(c->prec, AdjSmall{state(t), state(t - steps + 1), SZ / esz, mun, mu, c->flags, c->tb_lk, c->dsfrac, c->duin,
                                                     dJds, dJdu, win, m, c->tb_t, c->tb_k, steps, false}, fa, c->stream));
                    std::swap(mun, mu);
                    t -= steps;
                    continue;
                }
                AdjArgs aa;
                aa.f = fa;
                aa.alpha = win.at(m);
                aa.alpha_next = win.at(m + 1);
                ATRY(adj_step(Q, c->prec, state(t), mun, mu, c->flags, c->dsfrac, c->duin, dJds, dJdu, c->rowclean, c->adj_all_fast, aa,
                              c->stream));
                std::swap(mun, mu);
                t--;
            }
        }
        ATRY(adj_init(Q, c->prec, mun, c->flags, c->duin, dxi, c->cfg.perturb, c->cfg.seed, win.at(1),
                      dJdu, fa, c->stream));
    }
    ATRY(hipEventRecord(e2, c->stream));
    ATRY(hipEventSynchronize(e2));
    ATRY(hipEventElapsedTime(&tf, e0, e1));
    ATRY(hipEventElapsedTime(&ta, e1, e2));
    if (ms_forward) *ms_forward = tf;
    if (ms_adjoint) *ms_adjoint = ta;

    // ---- outputs ----
    if (J) {
        hist.resize(4 * (size_t)c->nrec);
        ATRY(hipMemcpy(hist.data(), c->hist, sizeof(double) * hist.size(), hipMemcpyDeviceToHost));
        double acc = 0.0;
        for (int r = 0; r < c->nrec; r++) acc += win.at((int)hist[4 * r]) * hist[4 * r + 1];
        *J = acc;
    }
    if (dJ_ds) {
        ATRY(hipMalloc(&tmp, sizeof(double) * c->N));
        ATRY(adj_reduce_ds(c->prec, dJds, tmp, g, c->stream));
        ATRY(hipMemcpyAsync(dJ_ds, tmp, sizeof(double) * c->N, hipMemcpyDeviceToHost, c->stream));
    }
    if (dJ_duin) ATRY(hipMemcpyAsync(dJ_duin, dJdu, sizeof(double) * g.ny * g.nz, hipMemcpyDeviceToHost, c->stream));
    ATRY(hipStreamSynchronize(c->stream));

done:
    c->cfg.force_interval = fi_saved;
    (void)hipStreamSynchronize(c->stream);
    for (void *p : {ckpt, store, mu0, mu1, (void *)dJds, (void *)dJdu, (void *)tmp, (void *)dxi})
        if (p) (void)hipFree(p);
    for (hipEvent_t e : {e0, e1, e2})
        if (e) (void)hipEventDestroy(e);
    return rc;
}
