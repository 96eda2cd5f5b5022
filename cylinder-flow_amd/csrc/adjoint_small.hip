// adjoint_small.hip -- several reverse steps per launch on the small D2Q9 domains that run several forward
// steps per launch (small_kernel.hpp), non-periodic.
//
// A reverse step of a 400x100 domain reads 6 MB, writes 3 and costs what a dependent launch costs (4.9 us).
// As forward: a block owns the W x W core of a T x T tile, holds mu of the tile in the LDS (two halves, one
// read and one written per step) and computes, per step, the nodes within the steps still to come of the
// core, the gather of mu_{m+1} being a plain LDS read: positions outside the domain and solid ones hold 0
// (inlet unknowns, beyond the outlet), and the links of the node's word take its own opposite value.  H_{m-1}
// is read from the stored states, pulled with the forward's rules, one step ahead of its use (its loads
// depend on nothing).  dJ/ds of the core and dJ/du_in of its inlet nodes stay in registers over the steps.
// Each node's arithmetic is k_adj_step's, so mu and the gradients equal its bit for bit.
#include "adjoint_common.hpp"
#include "small_kernel.hpp"

namespace lbm {

template <class S, int TB_T, bool SFRAC>
__global__ void __launch_bounds__((TB_T - 2) * (TB_T - 2))
    k_adj2d(const typename S::T *__restrict__ H, const typename S::T *__restrict__ Hlast, size_t stride, const typename S::C *__restrict__ mun,
            typename S::C *__restrict__ mu, const uint8_t *__restrict__ flags, const uint16_t *__restrict__ lk,
            const typename S::C *__restrict__ sfrac, const double *__restrict__ uin, double *__restrict__ dJds,
            double *__restrict__ dJdu, const FusedArgs a, AdjWindow win, int m, int K, int steps, int tiles_x, int ntiles) {
    using L = Lat<9>;
    using T = typename S::T;
    using C = typename S::C;
    constexpr int Q = 9, NT = (TB_T - 2) * (TB_T - 2), TP = tb_row(TB_T), HALF = Q * TB_T * TP;
    const Geo &g = a.g;
    const int W = TB_T - 2 * K;
    extern __shared__ __align__(16) char tb_lds[];
    C *const lds = (C *)tb_lds;
    const int t = threadIdx.x;
    const int tile = tb_tile_of_block(tiles_x, ntiles);
    int tx, ty;
    tb_place<TB_T>(t, K, tile % tiles_x == 0, tx, ty);
    const int dx = tx < K ? K - tx : (tx >= K + W ? tx - (K + W - 1) : 0);
    const int dy = ty < K ? K - ty : (ty >= K + W ? ty - (K + W - 1) : 0);
    const int slot = tx * TP + ty;
    const int X0 = (tile % tiles_x) * W - K, Y0 = (tile / tiles_x) * W - K;
    const int X = X0 + tx, Y = Y0 + ty;
    const bool in = X >= 0 && X < g.nx && Y >= 0 && Y < g.ny;
    const uint32_t ux = in ? (uint32_t)X : 0u, uy = in ? (uint32_t)Y : 0u, node = ux + (uint32_t)g.nxp * uy;
    const bool live = in && flags[node] != FL_SOLID;
    const int dist = live ? max(dx, dy) : TB_T;   // Chebyshev distance from the core; never computed otherwise
    const uint32_t w = lk[node];
    const bool xlo = X == 0, xhi = X == g.nx - 1;
    const C uy_in = (C)uin[uy];
    C sf = 0;
    if constexpr (SFRAC) sf = sfrac[node];
    const bool own = dist == 0, inlet = own && xlo;
    double ds = SFRAC && own ? dJds[node] : 0.0, du = inlet ? dJdu[uy] : 0.0;
    // the pull's links: bounced directions read the node's own opposite value; the gather along +e_i is
    // the pull of opp(i) reversed, except that beyond the outlet (whose pull is clamped to the outlet
    // column) there is nothing to gather
    const uint32_t solid = (w & 0xFFu) << 1, wall = (w >> 8) << 1;
    uint32_t off[Q];   // elements of H
    static_for<0, Q>([&](auto I) {
        constexpr int i = I;
        const bool own_row = ((solid | wall) >> i) & 1u;
        uint32_t sx = ux - (uint32_t)L::ex(i);
        const uint32_t sy = uy - (uint32_t)L::ey(i);
        if constexpr (L::ex(i) < 0) sx = xhi ? ux : sx;
        const bool unknown = L::ex(i) > 0 && xlo;   // at the inlet: read, then replaced
        off[i] = (own_row || unknown || !live) ? (uint32_t)pel(g, L::opp(i), ux, uy) : (uint32_t)pel(g, i, sx, sy);
    });
    constexpr uint32_t beyond = [] {   // the directions whose source the outlet clamps
        uint32_t b = 0;
        for (int i = 1; i < 9; i++)
            if (L::ex(i) < 0) b |= 1u << i;
        return b;
    }();
    const uint32_t gsolid = xhi ? solid & ~beyond : solid, gbounce = gsolid | wall;
    // mu of the tile, x fastest, into half 0; half 1 to 0
    for (int j = t; j < TB_T * TB_T; j += NT) {
        const int lx = j % TB_T, ly = j / TB_T, AX = X0 + lx, AY = Y0 + ly;
        const bool inside = AX >= 0 && AX < g.nx && AY >= 0 && AY < g.ny;
        const uint32_t ax = inside ? (uint32_t)AX : 0u, ay = inside ? (uint32_t)AY : 0u;
        C v[Q];
        static_for<0, Q>([&](auto I) { v[I] = mun[pel(g, I, ax, ay)]; });
        static_for<0, Q>([&](auto I) {
            lds[I * TB_T * TP + lx * TP + ly] = inside ? v[I] : (C)0;   // (solid nodes hold 0 in memory)
            lds[HALF + I * TB_T * TP + lx * TP + ly] = 0;
        });
    }
    T rh[Q] = {};
    if (dist <= steps - 1) static_for<0, Q>([&](auto I) { rh[I] = H[off[I]]; });   // (steps == 1: H is Hlast)
    C mm[Q] = {};
    for (int s = 0; s < steps; s++, m--) {
        lds_barrier();
        const C *const buf = lds + (s & 1) * HALF;
        C *const next = lds + (~s & 1) * HALF;
        const int rs = steps - 1 - s;
        C gv[Q];
        static_for<0, Q>([&](auto I) {
            constexpr int i = I;
            gv[i] = S::template decode<i, L>(rh[i], 0.f);
            if constexpr (L::ex(i) > 0) gv[i] = xlo ? (C)0 : gv[i];
        });
        if (dist < rs) {   // the next step's
            const T *const Hn = s + 2 == steps ? Hlast : H - stride * (size_t)(s + 1);
            static_for<0, Q>([&](auto I) { rh[I] = Hn[off[I]]; });
        }
        if (dist <= rs) {
            const double alpha = win.at(m);
            const C an = (C)win.at(m + 1);
            C lam[Q];
            static_for<0, Q>([&](auto I) {
                constexpr int i = I;
                constexpr int ex = L::ex(i), ey = L::ey(i), o = L::opp(i);
                C l = buf[i * TB_T * TP + slot + ex * TP + ey];
                if constexpr (i > 0) {
                    const C self = buf[o * TB_T * TP + slot];
                    if ((gbounce >> o) & 1u) l = ((gsolid >> o) & 1u) ? self + an * (C)(2 * ex) : self;
                }
                // the outlet node of row y + e_y pulls h_i from this node when e_ix < 0
                if constexpr (ex < 0) {
                    const C r = buf[i * TB_T * TP + slot + ey];
                    l = xhi ? l + r : l;
                }
                lam[i] = l;
            });
            if (xlo) velocity_inlet<Q, C>(gv, uy_in);
            double dds = 0.0;
            adj_transpose<Q, S, SFRAC>(lam, gv, sf, (C)a.rtau, alpha, mm, dds);
            if constexpr (SFRAC) ds += dds;   // (kept of the core's nodes alone)
            if (xlo) {
                double d = 0.0;
                adj_inlet_transpose<Q, S>(mm, d);
                du += d;
            }
            static_for<0, Q>([&](auto I) { next[I * TB_T * TP + slot] = mm[I]; });
        }
    }
    __syncthreads();
    if (SFRAC && own) dJds[node] = ds;
    if (inlet) dJdu[uy] = du;
    // the core, x fastest (solid nodes: 0 stays)
    const C *const out = lds + (steps & 1) * HALF;
    for (int j = t; j < W * W; j += NT) {
        const int lx = K + j % W, ly = K + j / W, AX = X0 + lx, AY = Y0 + ly;
        if (AX < g.nx && AY < g.ny)
            static_for<0, Q>([&](auto I) { mu[pel(g, I, (uint32_t)AX, (uint32_t)AY)] = out[I * TB_T * TP + lx * TP + ly]; });
    }
}

template <class S>
static hipError_t adj_small_s(const AdjSmall &l, const FusedArgs &a, hipStream_t s) {
    using T = typename S::T;
    using C = typename S::C;
    hipError_t e = hipErrorInvalidValue;
    int tiles_x = 0;
    const int ntiles = tb_tiles(a.g, l.T, l.K, &tiles_x);
    tb_side(l.T, [&](auto side) {
        constexpr int W = decltype(side)::value;
        const unsigned lds = (unsigned)(sizeof(C) * 2 * 9 * W * tb_row(W));
        auto go = [&](auto kern) {
            if (l.prepare) {
                e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
                return;
            }
            hipLaunchKernelGGL(kern, dim3((unsigned)ntiles), dim3((W - 2) * (W - 2)), lds, s, (const T *)l.H, (const T *)l.Hlast, l.stride,
                               (const C *)l.mun, (C *)l.mu, l.flags, l.lk, (const C *)l.sfrac, l.uin, l.dJds, l.dJdu, a, l.win, l.m,
                               l.K, l.steps, tiles_x, ntiles);
            e = hipGetLastError();
        };
        if (l.sfrac) go(k_adj2d<S, W, true>);
        else go(k_adj2d<S, W, false>);
    });
    return e;
}

hipError_t adj_small(int prec, const AdjSmall &l, const FusedArgs &a, hipStream_t s) {
    if (a.g.xper || a.g.yper || l.steps < 1 || l.steps > l.K || l.T - 2 * l.K < 1) return hipErrorInvalidValue;
    if (prec == LBM_FP64) return adj_small_s<SF64>(l, a, s);
    if (prec == LBM_FP32) return adj_small_s<SF32>(l, a, s);
    return hipErrorInvalidValue;
}

}  // namespace lbm
