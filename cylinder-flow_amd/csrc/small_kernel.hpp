// small_kernel.hpp -- several D2Q9 steps per launch for small domains (plain mode).
//
// On a 400x100 domain one step moves 5.8 MB and the kernel itself takes about a microsecond,
// so a step costs what a dependent launch costs (~3.4 us on one MI355X; a captured graph of
// launches costs the same).  Temporal blocking removes all but one launch per K steps: block b
// owns a W x W core of nodes and loads its core plus a halo of K nodes on each side (T x T
// nodes, T = 24..32, K and T chosen for the domain by tb_choose) into the LDS,
// coalesced; each of the K steps pulls from the LDS (boundary rules applied by the values the
// live nodes write, setup_links9) and collides in registers (one thread per node), and the live
// nodes write their populations back to the LDS.  A halo node's result is exact as long as every node it pulled from was, so the exact
// region shrinks by one node per step and after K steps covers the core, which is written out;
// each step computes only that region (threads in ring order, the waves outside it idle).  No
// block reads another block's output within a launch: there is no grid-wide synchronisation.
// Each node's arithmetic is that of the one-step kernels (same pull classification, inlet,
// collide_f64 or collide, the storage format's decode and encode; the LDS holds stored values), so
// the populations equal the one-launch-per-step path bit for bit; forces are summed per tile (a
// different summation order than the per-row blocks of k_fused and k_dense_v, the same value to
// rounding).
#pragma once
#include "fast_kernel.hpp"

namespace lbm {

constexpr int TB_KMAX = 10;   // steps per launch at most (tb_choose)

// LDS row length (doubles) of a T x T tile: the odd one of T + 1, T + 2
__host__ __device__ constexpr int tb_row(int T) { return T % 2 == 0 ? T + 1 : T + 2; }

// Threads take the tile's nodes ring by ring from the core outwards: threads [0, W*W) the
// core (y fastest), then ring r = 1..K-1 (the nodes at Chebyshev distance r from the core:
// its left and right columns, then its top and bottom rows).  The nodes a step must compute,
// the live nodes within the steps still to come of the core, are then the first (W + 2m)^2
// threads, and the waves beyond them skip the step: the busiest SIMD of a 24 x 24 tile runs
// 2+2+2+1+1 wave-steps in 5 steps instead of 3 per step.  Tiles at the inlet (their left K
// columns lie outside the domain) take the inlet column x = 0 first, so that one wave runs
// the inlet's long sequence, then the nodes right of it ring by ring, then those left of it
// (never computed).
template <int TB_T>
__device__ __forceinline__ void tb_place(int t, int K, bool inlet, int &tx, int &ty) {
    const int W = TB_T - 2 * K;
    if (!inlet) {
        if (t < W * W) {
            tx = K + t / W;
            ty = K + t % W;
        } else {
            int r = 1, side = W + 2;
            while (t >= side * side) {   // at most K - 1 rings: blockDim.x is NT
                r++;
                side += 2;
            }
            const int q = t - (side - 2) * (side - 2), lo = K - r, hi = lo + side - 1;
            if (q < side) {
                tx = lo;
                ty = lo + q;
            } else if (q < 2 * side) {
                tx = hi;
                ty = lo + q - side;
            } else if (q < 3 * side - 2) {
                ty = lo;
                tx = lo + 1 + q - 2 * side;
            } else {
                ty = hi;
                tx = lo + 1 + q - (3 * side - 2);
            }
        }
    } else {
        int q = t;
        if (q < TB_T - 2) {                      // the inlet column
            tx = K;
            ty = 1 + q;
        } else if ((q -= TB_T - 2) < (W - 1) * W) {   // the core right of it
            tx = K + 1 + q / W;
            ty = K + q % W;
        } else {
            q -= (W - 1) * W;
            int r = 1;
            while (r < K && q >= 3 * W + 4 * r - 4) {  // ring r right of the inlet column
                q -= 3 * W + 4 * r - 4;
                r++;
            }
            if (r < K) {
                if (q < W + 2 * r) {                   // its right column
                    tx = K + W - 1 + r;
                    ty = K - r + q;
                } else if ((q -= W + 2 * r) < W + r - 2) {   // its top row
                    ty = K - r;
                    tx = K + 1 + q;
                } else {                               // its bottom row
                    ty = K + W - 1 + r;
                    tx = K + 1 + q - (W + r - 2);
                }
            } else {                                   // left of the inlet column
                tx = 1 + q / (TB_T - 2);
                ty = 1 + q % (TB_T - 2);
            }
        }
    }
}

// Workgroups go to the 8 XCDs in turn (b % 8), each XCD with its own L2: XCD k takes the
// consecutive positions [k (n / 8) + min(k, n % 8), ...) of the n = ntiles in an order that
// runs down bands of two tile rows column by column, so that an XCD holds a 2-row block of
// neighbouring tiles, whose loads overlap, read through one L2 (on 400 x 100, 2 x 14-15
// tiles per XCD: 10 % fewer microseconds per step than neighbouring tiles on different XCDs)
__device__ __forceinline__ int tb_tile_of_block(int tiles_x, int ntiles) {
    const int xcd = (int)(blockIdx.x % 8u);
    const int pos = xcd * (ntiles / 8) + min(xcd, ntiles % 8) + (int)(blockIdx.x / 8u);
    const int band = pos / (2 * tiles_x), in_band = pos % (2 * tiles_x);
    const int band_rows = min(2, ntiles / tiles_x - 2 * band);
    return (2 * band + in_band % band_rows) * tiles_x + in_band / band_rows;
}

template <class S, int TB_T, bool ANY_FORCE, bool SFRAC>
__global__ void __launch_bounds__(1024)
    k_tb2d(const typename S::T *__restrict__ A, typename S::T *__restrict__ B, const uint8_t *__restrict__ flags,
           const uint16_t *__restrict__ lk, const typename S::C *__restrict__ sfrac, const double *__restrict__ uin,
           double *__restrict__ partials, typename S::T *__restrict__ keep, size_t keep_stride,
           const FusedArgs a, int K, int steps, long step0, int fi, int tiles_x, int ntiles, int pend) {
    using L = Lat<9>;
    using T = typename S::T;
    using C = typename S::C;
    // one thread per node of the rings a step can compute (within K - 1 of the core); the
    // outermost ring is only read, and is loaded with the rest of the tile
    constexpr int Q = 9, NT = (TB_T - 2) * (TB_T - 2);
    static_assert((NT + 63) / 64 <= 16, "force records hold 16 waves");
    const Geo &g = a.g;
    const int W = TB_T - 2 * K;          // core side
    // LDS: two halves of Q x TB_T x TP values (step s reads half s % 2; node (tx, ty) at
    // tx * TP + ty, rows padded to the odd TP = tb_row(TB_T) so that lanes TP apart hit different
    // banks: an even row of 32 doubles puts every x of a row segment on one bank),
    // then the tile's link words (TB_T x TP) and flags (TB_T x TP bytes)
    constexpr int TP = tb_row(TB_T), HALF = Q * TB_T * TP;
    extern __shared__ __align__(16) char tb_lds[];
    T *const lds = (T *)tb_lds;
    uint16_t *llk = (uint16_t *)(lds + 2 * HALF);
    uint8_t *lfl = (uint8_t *)(llk + TB_T * TP);
    const int t = threadIdx.x;
    const int tile = tb_tile_of_block(tiles_x, ntiles);
    int tx, ty;
    tb_place<TB_T>(t, K, tile % tiles_x == 0, tx, ty);
    // Chebyshev distance of the node from the core
    const int dx = tx < K ? K - tx : (tx >= K + W ? tx - (K + W - 1) : 0);
    const int dy = ty < K ? K - ty : (ty >= K + W ? ty - (K + W - 1) : 0);
    const int dist = dx > dy ? dx : dy;
    const int slot = tx * TP + ty;       // LDS index of the node
    const int X0 = (tile % tiles_x) * W - K, Y0 = (tile / tiles_x) * W - K;
    const int X = X0 + tx, Y = Y0 + ty;
    const bool act = X >= 0 && X < g.nx && Y >= 0 && Y < g.ny;
    const bool own = act && tx >= K && tx < K + W && ty >= K && ty < K + W;
    const C uy = (C)uin[act ? Y : 0];
    C sfv = 0;
    if constexpr (SFRAC) sfv = act ? sfrac[(uint32_t)X + (uint32_t)g.nxp * (uint32_t)Y] : (C)0;
    // Every pull is a plain LDS read at the source's position (no boundary rule in the pull):
    // each live node also writes, with its own values, the values its rules pull from
    // positions no live node owns: h_opp(i) into the source position of each bounce-back link i
    // (a wall or a solid source, from its link word: only this node pulls direction i from
    // there), and at the outlet (x = nx - 1) its values of the directions with e_x < 0 into the
    // position beyond the outlet (x = nx), which the outlet node above or below pulls for the
    // zero gradient.  The inlet's unknowns read positions left of the inlet, which hold 0.
    // The tile's link words, flags and populations, x fastest (coalesced), into the LDS (into
    // half 0 with the first step's ghost values, which the loading thread writes for its node;
    // half 1's positions outside the domain to 0): node t, t + NT, ... of the tile's T*T, every
    // load issued (from node (0, 0) for positions outside the domain) before the first is used.
    {
        constexpr int NJ = (TB_T * TB_T + NT - 1) / NT;
        T v[NJ][Q];
        uint8_t f[NJ];
        uint16_t w[NJ];
#pragma unroll
        for (int k = 0; k < NJ; k++) {
            const int j = t + k * NT, lx = j % TB_T, ly = j / TB_T, AX = X0 + lx, AY = Y0 + ly;
            const bool in = j < TB_T * TB_T && AX >= 0 && AX < g.nx && AY >= 0 && AY < g.ny;
            const uint32_t ax = in ? (uint32_t)AX : 0u, ay = in ? (uint32_t)AY : 0u, node = ax + (uint32_t)g.nxp * ay;
            f[k] = flags[node];
            w[k] = lk[node];
            static_for<0, Q>([&](auto I) { v[k][I] = A[pel(g, I, ax, ay)]; });
        }
#pragma unroll
        for (int k = 0; k < NJ; k++) {
            const int j = t + k * NT, lx = j % TB_T, ly = j / TB_T, AX = X0 + lx, AY = Y0 + ly;
            const bool in = AX >= 0 && AX < g.nx && AY >= 0 && AY < g.ny;
            if (j < TB_T * TB_T) {
                const int pos = lx * TP + ly;
                const bool lv = in && f[k] != FL_SOLID;
                lfl[pos] = in ? f[k] : (uint8_t)FL_SOLID;
                llk[pos] = lv ? w[k] : (uint16_t)0;
                if (lv) {
                    static_for<0, Q>([&](auto I) { lds[I * TB_T * TP + pos] = v[k][I]; });
                    const uint32_t bbk = ((uint32_t)(w[k] & 0xFFu) | (uint32_t)(w[k] >> 8)) << 1;
                    if (bbk != 0u)
                        static_for<1, Q>([&](auto I) {
                            constexpr int i = I;
                            constexpr int ex = L::ex(i), ey = L::ey(i), o = L::opp(i);
                            // positions beyond the tile feed only its outermost ring, never computed
                            if (((bbk >> i) & 1u) && (unsigned)(lx - ex) < (unsigned)TB_T &&
                                (unsigned)(ly - ey) < (unsigned)TB_T)
                                lds[i * TB_T * TP + pos - ex * TP - ey] = v[k][o];
                        });
                    if (AX == g.nx - 1 && lx + 1 < TB_T)
                        static_for<1, Q>([&](auto I) {
                            constexpr int i = I;
                            if constexpr (L::ex(i) < 0) lds[i * TB_T * TP + pos + TP] = v[k][i];
                        });
                }
                if (AX < 0) static_for<0, Q>([&](auto I) { lds[I * TB_T * TP + pos] = T(0); });
                if (!in) static_for<0, Q>([&](auto I) { lds[HALF + I * TB_T * TP + pos] = T(0); });
            }
        }
    }
    __syncthreads();
    const uint8_t fl = lfl[slot];
    const bool live = fl != FL_SOLID;
    const uint32_t lkw = llk[slot];
    const uint32_t solid_src = (lkw & 0xFFu) << 1;                 // mask links (momentum exchange)
    const uint32_t bb = solid_src | ((lkw >> 8) << 1);              // every bounce-back link
    const bool outl = live && X == g.nx - 1;
    // a node's values in registers: every step pulls from the LDS, and a node writes (from the
    // second step on, and into the core store) only values a step of its own computed
    T h[Q] = {};
    // force records: the steps s = sf, sf + fi, ... of this launch (step0 + s + 1 a multiple of
    // fi); each wave's sums go to red[record][wave] and are added, waves in order, after the
    // launch's last barrier, so no force step waits for a block-wide sum
    __shared__ double red[3 * 16 * TB_KMAX];
    int sf = ANY_FORCE && fi > 0 ? (int)(fi - 1 - step0 % fi) : -1, kr = 0;
    auto store_core = [&](const T *from, T *to) {   // x fastest
        for (int j = t; j < W * W; j += NT) {
            const int lx = K + j % W, ly = K + j / W, AX = X0 + lx, AY = Y0 + ly;
            if (AX < g.nx && AY < g.ny && lfl[lx * TP + ly] != FL_SOLID)
                static_for<0, Q>([&](auto I) {
                    __builtin_nontemporal_store(from[I * TB_T * TP + lx * TP + ly], &to[pel(g, I, (uint32_t)AX, (uint32_t)AY)]);
                });
        }
    };
    for (int s = 0; s < steps; s++) {
        const bool force = ANY_FORCE && s == sf;
        // two halves: the barrier of step s also orders the reads of step s - 1 before the writes
        // of step s + 1 into the same half
        T *buf = lds + (size_t)(s & 1) * HALF;
        // this step computes the live nodes within rs = steps - 1 - s of the core, from the
        // values of those within rs + 1 (computed by the previous step, or loaded into half 0
        // with the ghost values)
        const int rs = steps - 1 - s;
        if (s > 0) {
            if (dist <= rs + 1 && live) {
                static_for<0, Q>([&](auto I) { buf[I * TB_T * TP + slot] = h[I]; });
                if (bb != 0u)
                    static_for<1, Q>([&](auto I) {
                        constexpr int i = I;
                        constexpr int ex = L::ex(i), ey = L::ey(i), o = L::opp(i);
                        if ((bb >> i) & 1u) buf[i * TB_T * TP + slot - ex * TP - ey] = h[o];
                    });
                if (outl)
                    static_for<1, Q>([&](auto I) {
                        constexpr int i = I;
                        if constexpr (L::ex(i) < 0) buf[i * TB_T * TP + slot + TP] = h[i];
                    });
            }
            __syncthreads();
            if constexpr (!ANY_FORCE)   // (states are kept without force records)
                if (keep != nullptr) store_core(buf, keep + keep_stride * (size_t)(s - 1));
        }
        double fx = 0.0, fy = 0.0;
        if (dist <= rs && live) {
            C gv[Q];
            static_for<0, Q>([&](auto I) {
                constexpr int i = I;
                gv[i] = S::template decode<i, L>(buf[i * TB_T * TP + slot - L::ex(i) * TP - L::ey(i)], 0.f);
            });
            // momentum exchange of the mask links, in direction order, from the pulled values
            // (before the inlet rule), outside the pull so the other steps run without it
            if (ANY_FORCE && force && solid_src != 0u) {
                static_for<1, Q>([&](auto I) {
                    constexpr int i = I;
                    constexpr int ex = L::ex(i), ey = L::ey(i);
                    if ((solid_src >> i) & 1u) {
                        const double m = 2.0 * (double)gv[i];
                        if constexpr (ex != 0) fx -= ex * m;
                        if constexpr (ey != 0) fy -= ey * m;
                    }
                });
            }
            if (X == 0 && live) velocity_inlet<Q, C>(gv, uy);
            C c[Q], p, u, v, w;
            double fz = 0.0, sx = 0.0, sy = 0.0;
            if constexpr (sizeof(C) == 8) collide_f64<Q, ANY_FORCE, SFRAC>(gv, sfv, a.tau, a.rtau, c, p, u, v, w, sx, sy, fz);
            else collide<Q, ANY_FORCE, SFRAC>(gv, sfv, a.omega, c, p, u, v, w, sx, sy, fz);
            if constexpr (ANY_FORCE && SFRAC) {   // the solid fraction's force of a recorded step
                if (force) {
                    fx += sx;
                    fy += sy;
                }
            }
            static_for<0, Q>([&](auto I) { h[I] = S::template enc<I, L>(c[I], StoreParams{}); });
        }
        if (ANY_FORCE && force) {   // uniform over the grid
            double fz = 0.0;
            if (!own) fx = fy = 0.0;
            wave_sum3(fx, fy, fz);
            if ((t & 63) == 0) {
                double *R = red + 3 * (16 * kr + (t >> 6));
                R[0] = fx;
                R[1] = fy;
                R[2] = fz;
            }
            kr++;
            sf += fi;
        }
    }
    // the core through the LDS half the last step did not read (its last reader, step
    // steps - 2, finished before the barrier of step steps - 1), then stored x fastest
    T *out = lds + (size_t)(steps & 1) * HALF;
    if (dist == 0) static_for<0, Q>([&](auto I) { out[I * TB_T * TP + slot] = h[I]; });
    __syncthreads();
    if (ANY_FORCE && t < kr) {
        // record t of this launch into slot pend + t: the waves' sums in wave order
        constexpr int NW = (NT + 63) / 64;
        const double *R = red + 3 * 16 * t;
        double fx = R[0], fy = R[1], fz = R[2];
        for (int k = 1; k < NW; k++) {
            fx += R[3 * k];
            fy += R[3 * k + 1];
            fz += R[3 * k + 2];
        }
        double *P = partials + 3 * ((size_t)(pend + t) * ntiles + tile);
        P[0] = fx;
        P[1] = fy;
        P[2] = fz;
    }
    store_core(out, B);
}

// ---- launchers of one storage format (small_f64.hip ... small_bf16.hip) ----
// LDS row length of a T x T tile and its LDS bytes for values of esz bytes: two population halves of
// 9 x T x tb_row(T) values, the tile's link words and flags (T x tb_row(T) of each)
inline size_t tb_lds_size(int T, size_t esz) { return esz * 2 * 9 * T * tb_row(T) + (size_t)3 * T * tb_row(T); }

struct TbLaunch {
    const void *A;
    void *B;
    const uint8_t *flags;
    const uint16_t *lk;
    const void *sfrac;
    const double *uin;
    double *partials;
    void *keep;            // null, or where the states before the last go, keep_stride elements apart
    size_t keep_stride;
    int T, K, steps, fi, tiles_x, ntiles, pend;
    long step0;
    bool force;
    bool prepare;   // only set the kernel's LDS limit on the current device (before its first launch there)
};

// f(std::integral_constant<int, T>) for the instantiated tile side T; false: not instantiated
template <class F>
static bool tb_side(int T, F &&f) {
    bool hit = false;
    auto one = [&](auto t) {
        if (T == decltype(t)::value) {
            f(t);
            hit = true;
        }
    };
    one(std::integral_constant<int, 24>{});
    one(std::integral_constant<int, 25>{});
    one(std::integral_constant<int, 26>{});
    one(std::integral_constant<int, 27>{});
    one(std::integral_constant<int, 28>{});
    one(std::integral_constant<int, 29>{});
    one(std::integral_constant<int, 30>{});
    one(std::integral_constant<int, 31>{});
    one(std::integral_constant<int, 32>{});
    return hit;
}

template <class S>
static hipError_t tb_launch_s(const TbLaunch &l, const FusedArgs &a, hipStream_t s) {
    using T = typename S::T;
    hipError_t e = hipErrorInvalidValue;
    const size_t lds = tb_lds_size(l.T, sizeof(T));
    tb_side(l.T, [&](auto side) {
        constexpr int W = decltype(side)::value;
        auto go = [&](auto kern) {   // (T - 2)^2 threads: the kernel's thread map assumes exactly that
            if (l.prepare) {
                e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
                return;
            }
            hipLaunchKernelGGL(kern, dim3(l.ntiles), dim3((W - 2) * (W - 2)), lds, s, (const T *)l.A, (T *)l.B, l.flags, l.lk,
                               (const typename S::C *)l.sfrac, l.uin, l.partials, (T *)l.keep, l.keep_stride, a, l.K, l.steps, l.step0, l.fi, l.tiles_x,
                               l.ntiles, l.pend);
            e = hipGetLastError();
        };
        if (l.sfrac) l.force ? go(k_tb2d<S, W, true, true>) : go(k_tb2d<S, W, false, true>);
        else l.force ? go(k_tb2d<S, W, true, false>) : go(k_tb2d<S, W, false, false>);
    });
    return e;
}

}  // namespace lbm
