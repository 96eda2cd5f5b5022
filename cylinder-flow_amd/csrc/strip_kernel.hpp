// strip_kernel.hpp -- several D2Q9 steps per pass over memory on large domains (plain mode, every
// storage format).
//
// One step moves 18 values per node for about 110 instructions of arithmetic, and is bound by HBM.
// k_strip advances the state by K steps per launch and moves those values once.  Every wave works
// alone, without LDS or barriers: its 64 lanes are 64 neighbouring columns, and it marches along y.
// In a pass, the first step's row p is pulled from A (boundary rules in the lane's offsets and the
// bounce words), and step l + 1 completes row p - l from what step l has just left in registers:
// the directions with e_x != 0 come from the neighbouring lane (a wave shift), those with e_y = +1
// wait one pass, as in the D3Q27 kernel of pair_kernel.hpp, which is organised the same way.  Each
// step loses one column at either end of the wave, so step K is valid on 66 - 2K columns, which are
// stored; the rows above and below a run of rows are recomputed by both neighbours.
// 2048 x 2048, drag every 10 steps, us per step, one step per launch / four per pass: FP64 100.7 / 57.8,
// FP32 50.7 / 24.9, FP16 27.2 / 23.5; 8192 x 4096: 809 / 417, 384 / 202, 206 / 146.  Bound by
// instruction issue (460 vector instructions per wave and row of four steps, 1.3 times the work in
// rims), so it is HBM no longer; a run of rows per resident wave (2 per SIMD in FP64, 4 otherwise)
// measured best: 28.2 / 25.5 / 25.1 / 27.0 in FP32 at 2 / 3 / 4 / 6 per SIMD.
//
// Stored values are rounded to the storage format between the steps and every node's arithmetic is
// that of the one-step kernels, so populations are theirs bit for bit; force records are summed per
// wave and then over the waves (the same value to rounding).
#pragma once
#include "pair_kernel.hpp"

namespace lbm {

// value of the lane to the left (SH = +1) or right (SH = -1); the end lanes keep a value of their own
template <int SH, class T>
__device__ __forceinline__ T lane_shift(T v) {
    constexpr int ctrl = SH > 0 ? 0x138 : 0x130;   // wave_shr:1, wave_shl:1
    if constexpr (sizeof(T) == 8) {
        int u[2];
        __builtin_memcpy(u, &v, 8);
        u[0] = __builtin_amdgcn_update_dpp(u[0], u[0], ctrl, 0xf, 0xf, false);
        u[1] = __builtin_amdgcn_update_dpp(u[1], u[1], ctrl, 0xf, 0xf, false);
        __builtin_memcpy(&v, u, 8);
    } else {
        typename UInt<sizeof(T)>::type b;
        __builtin_memcpy(&b, &v, sizeof(T));
        b = (decltype(b))__builtin_amdgcn_update_dpp((int)b, (int)b, ctrl, 0xf, 0xf, false);
        __builtin_memcpy(&v, &b, sizeof(T));
    }
    return v;
}

// rank of direction i among the D2Q9 directions with its e_y
constexpr int yrank(int i) {
    int k = 0;
    for (int j = 0; j < i; j++) k += Lat<9>::ey(j) == Lat<9>::ey(i);
    return k;
}

template <class S, int K, bool FORCE, bool SFRAC>
struct StripMarch {
    using L = Lat<9>;
    using T = typename S::T;
    using C = typename S::C;
    static constexpr int Q = 9;
    static_assert(K >= 2 && K <= 8, "steps per pass");
    typedef const __attribute__((address_space(4))) double *cdouble;

    const FusedArgs &a;
    cdouble uin;
    __amdgpu_buffer_rsrc_t in, out, words, solid;
    uint32_t rsb, dsb;              // bytes of a row and of a direction within it
    uint32_t co[3], outx, wx, sx;   // lane offsets: columns e_x = -1, 0, +1; store; bounce word; solid fraction
    bool core, inlet, outlet;       // lane's column: stored, x = 0, x = nx - 1
    bool has_inlet, has_outlet;     // in the wave
    int y0, y1;
    uint32_t rec;                   // bit l: step l + 1 records the force

    T R[Q];                          // raw populations of the next row (in flight)
    uint32_t wn;                     // its bounce word, and the words of rows p, p - 1, ...
    uint32_t W[K];
    C sn, SF[SFRAC ? K : 1];
    T up[K - 1][3], mid[K - 1][3], upn[K - 1][3], own[K - 1][3];   // step l + 2: see pair_kernel.hpp
    double fx[FORCE ? K : 1], fy[FORCE ? K : 1];

    __device__ __forceinline__ int wrapy(int y) const {
        const int n = a.g.ny, c = min(max(y, 0), n - 1), w = y + (y < 0 ? n : 0) - (y >= n ? n : 0);
        return __builtin_amdgcn_readfirstlane(a.g.yper ? min(max(w, 0), n - 1) : c);
    }
    __device__ __forceinline__ static bool any(bool b) { return __builtin_amdgcn_ballot_w64(b) != 0ull; }

    // bounced directions of a word: mask links in its low byte, walls in its high byte
    __device__ __forceinline__ static uint32_t bounced(uint32_t w) { return ((w & 0xffu) | (w >> 8)) << 1; }

    __device__ __forceinline__ void issue(int y) {
        const int yy = wrapy(y), ym = wrapy(yy - 1), yp = wrapy(yy + 1);
        const uint32_t s0 = rsb * (uint32_t)yy, sm = rsb * (uint32_t)ym, sp = rsb * (uint32_t)yp;
        const uint32_t w = bounced(wn);   // of row y, loaded one pass before
        W[0] = wn;
        if constexpr (SFRAC) {
            SF[0] = sn;
            sn = buf_load<C>(solid, sx, (uint32_t)sizeof(C) * (uint32_t)a.g.nxp * (uint32_t)wrapy(y + 1));
        }
        wn = buf_load<uint16_t>(words, wx, 2u * (uint32_t)a.g.nxp * (uint32_t)wrapy(y + 1));
        if (any(w != 0u)) {
            static_for<0, Q>([&](auto I) {
                constexpr int i = I;
                const uint32_t nom = co[L::ex(i) + 1] + ((L::ey(i) > 0 ? sm : L::ey(i) < 0 ? sp : s0) + i * dsb);
                const uint32_t own_ = co[1] + (s0 + L::opp(i) * dsb);
                R[i] = buf_load<T>(in, pair_pick<uint32_t>(w, i, own_, nom), 0);
            });
        } else {
            static_for<0, Q>([&](auto I) {
                constexpr int i = I;
                R[i] = buf_load<T>(in, co[L::ex(i) + 1], (L::ey(i) > 0 ? sm : L::ey(i) < 0 ? sp : s0) + i * dsb);
            });
        }
    }

    // step l + 1 of row y: from the pulled values g to the stored values h
    template <int l>
    __device__ __forceinline__ void update(int y, C *g, T *h) {
        if constexpr (FORCE) {
            // momentum exchange of the mask links of the run's own nodes, before the inlet rule
            const uint32_t m = core ? (W[l] & 0xffu) << 1 : 0u;
            if (((rec >> l) & 1u) && y >= y0 && y < y1 && any(m != 0u))
                static_for<1, Q>([&](auto I) {
                    constexpr int i = I;
                    if ((m >> i) & 1u) {
                        const double e = 2.0 * (double)g[i];
                        if constexpr (L::ex(i) != 0) fx[l] -= L::ex(i) * e;
                        if constexpr (L::ey(i) != 0) fy[l] -= L::ey(i) * e;
                    }
                });
        }
        if (has_inlet) {
            const C U = (C)uin[wrapy(y)];
            if (inlet) velocity_inlet<Q, C>(g, U);
        }
        C c[Q], s, u, v, w;
        double sx_ = 0.0, sy_ = 0.0, sz_ = 0.0;
        const C sf = SFRAC ? SF[SFRAC ? l : 0] : (C)0;
        if constexpr (sizeof(C) == 8) collide_f64<Q, FORCE, SFRAC>(g, sf, a.tau, a.rtau, c, s, u, v, w, sx_, sy_, sz_);
        else collide<Q, FORCE, SFRAC>(g, sf, a.omega, c, s, u, v, w, sx_, sy_, sz_);
        if constexpr (FORCE && SFRAC)
            if (((rec >> l) & 1u) && y >= y0 && y < y1) {
                fx[l] += core ? sx_ : 0.0;
                fy[l] += core ? sy_ : 0.0;
            }
        static_for<0, Q>([&](auto I) { h[I] = S::template enc<I, L>(c[I], StoreParams{}); });
    }

    // h (step l of row y): completes step l + 1's row y - 1, whose values replace h, and collects what
    // row y and row y + 1 take from it
    template <int l>
    __device__ __forceinline__ void level(int y, T *h) {
        T sh[Q], r[Q];   // what this lane pulls of row y
        static_for<0, Q>([&](auto I) {
            constexpr int i = I;
            if constexpr (L::ex(i) > 0) sh[i] = lane_shift<1>(h[i]);
            else if constexpr (L::ex(i) < 0) sh[i] = lane_shift<-1>(h[i]);
            else sh[i] = h[i];
        });
        if (has_outlet)   // zero gradient: the outlet column takes its own
            static_for<0, Q>([&](auto I) {
                constexpr int i = I;
                if constexpr (L::ex(i) < 0) sh[i] = outlet ? h[i] : sh[i];
            });
        static_for<0, Q>([&](auto I) {
            constexpr int i = I;
            if constexpr (L::ey(i) > 0) r[i] = up[l - 1][yrank(i)];
            else if constexpr (L::ey(i) == 0) r[i] = mid[l - 1][yrank(i)];
            else r[i] = sh[i];
        });
        const uint32_t wj = bounced(W[l]), wk = bounced(W[l - 1]);   // rows y - 1 and y
        if (any(wj != 0u))
            static_for<1, Q>([&](auto I) {
                constexpr int i = I;
                if constexpr (L::ey(i) < 0) r[i] = pair_pick<T>(wj, i, own[l - 1][yrank(L::opp(i))], r[i]);
            });
        static_for<0, Q>([&](auto I) {
            constexpr int i = I;
            if constexpr (L::ey(i) > 0) {
                up[l - 1][yrank(i)] = upn[l - 1][yrank(i)];
                upn[l - 1][yrank(i)] = sh[i];
                own[l - 1][yrank(i)] = h[i];
            } else if constexpr (L::ey(i) == 0) {
                mid[l - 1][yrank(i)] = sh[i];
            }
        });
        if (any(wk != 0u))
            static_for<1, Q>([&](auto I) {
                constexpr int i = I;
                if constexpr (L::ey(i) > 0) up[l - 1][yrank(i)] = pair_pick<T>(wk, i, h[L::opp(i)], up[l - 1][yrank(i)]);
                else if constexpr (L::ey(i) == 0) mid[l - 1][yrank(i)] = pair_pick<T>(wk, i, h[L::opp(i)], mid[l - 1][yrank(i)]);
            });
        C g[Q];
        static_for<0, Q>([&](auto I) { g[I] = S::template decode<I, L>(r[I], 0.f); });
        update<l>(y - 1, g, h);
    }

    __device__ __forceinline__ void run() {
        static_for<0, Q>([&](auto I) { R[I] = T(0); });
        static_for<0, K>([&](auto I) { W[I] = 0u; });
        if constexpr (FORCE) static_for<0, K>([&](auto I) { fx[I] = fy[I] = 0.0; });
        static_for<0, K - 1>([&](auto J) {
            static_for<0, 3>([&](auto I) { up[J][I] = mid[J][I] = upn[J][I] = own[J][I] = T(0); });
        });
        if (y0 >= y1) return;   // the second half of a short last run
        const int first = y0 - (K - 1);
        const int fy_ = wrapy(first);
        wn = buf_load<uint16_t>(words, wx, 2u * (uint32_t)a.g.nxp * (uint32_t)fy_);
        if constexpr (SFRAC) {
            static_for<0, K>([&](auto I) { SF[I] = (C)0; });
            sn = buf_load<C>(solid, sx, (uint32_t)sizeof(C) * (uint32_t)a.g.nxp * (uint32_t)fy_);
        }
        issue(first);
        for (int p = first; p < y1 + K - 1; p++) {
            C g[Q];
            T h[Q];
            static_for<0, Q>([&](auto I) { g[I] = pinned<C>(S::template decode<I, L>(R[I], 0.f)); });
            const uint32_t w0 = W[0];
            const C s0 = SF[0];
            __builtin_amdgcn_sched_barrier(0);
            issue(p + 1 < y1 + K - 1 ? p + 1 : p);
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t w1 = W[0];
            const C s1 = SF[0];
            W[0] = w0;   // this pass's row
            SF[0] = s0;
            update<0>(p, g, h);
            // step l + 1's row p - l is first needed from row y0 - (K - 1 - l) on, and what it takes from
            // step l two rows before: earlier passes do nothing
            static_for<1, K>([&](auto J) {
                constexpr int l = J;
                if (l == K - 1 || p >= first + 2 * l - 2) level<l>(p - l + 1, h);
            });
            const int y = p - (K - 1);
            const uint32_t row = (uint32_t)(y >= y0 ? y : y0);
            static_for<0, Q>([&](auto I) { buf_store<T>(out, y >= y0 ? outx : ~0u, row * rsb + (uint32_t)I * dsb, h[I]); });
            static_for<1, K>([&](auto J) {   // W[j]: row p + 1 - j of the next pass
                constexpr int j = K - J;
                W[j] = W[j - 1];
                if constexpr (SFRAC) SF[j] = SF[j - 1];
            });
            W[0] = w1;
            SF[0] = s1;
        }
    }
};

template <class S, int K, bool FORCE, bool SFRAC>
__global__ void __launch_bounds__(256)
    k_strip(const typename S::T *__restrict__ A, typename S::T *__restrict__ B, const uint16_t *__restrict__ lk,
            const typename S::C *__restrict__ sfrac, const double *__restrict__ uin, double *__restrict__ partials,
            const FusedArgs a, int strips, int rows, int nwaves, uint32_t rec, int pend) {
    using T = typename S::T;
    const Geo &g = a.g;
    constexpr int WC = 66 - 2 * K;
    // workgroups go to the 8 XCDs in turn: each takes a run of neighbouring strips (four per group)
    const int n = (int)gridDim.x, xcd = (int)(blockIdx.x % 8u);
    const int pos = xcd * (n / 8) + min(xcd, n % 8) + (int)(blockIdx.x / 8u);
    const int wave = __builtin_amdgcn_readfirstlane(pos * 4 + (int)(threadIdx.x >> 6));
    if (wave >= nwaves) return;
    // the strip at the inlet, whose waves run the inlet's rule in every step, is two waves of half the rows
    const int split = g.xper ? 0 : 1, per_run = strips + split;
    const int run = __builtin_amdgcn_readfirstlane(wave / per_run), v = wave - run * per_run, strip = max(v - split, 0);
    const int lane = (int)(threadIdx.x & 63u), X0 = strip * WC;
    int X = X0 - (K - 1) + lane;
    const bool inside = g.xper || (X >= 0 && X < g.nx);
    if (g.xper) X = X < 0 ? (X + g.nx * ((-X + g.nx - 1) / g.nx)) : X % g.nx;
    X = min(max(X, 0), g.nx - 1);
    const uint32_t esz = (uint32_t)sizeof(T);
    const size_t bytes = sizeof(T) * 9 * g.plane;
    StripMarch<S, K, FORCE, SFRAC> m{a};
    m.uin = (typename StripMarch<S, K, FORCE, SFRAC>::cdouble)(uintptr_t)uin;
    m.in = plane_rsrc(A, (uint32_t)bytes);
    m.out = plane_rsrc(B, (uint32_t)bytes);
    m.words = plane_rsrc(lk, (uint32_t)(2 * g.plane));
    if constexpr (SFRAC) m.solid = plane_rsrc(sfrac, (uint32_t)(sizeof(typename S::C) * g.plane));
    m.rsb = (uint32_t)g.rs * esz;
    m.dsb = (uint32_t)g.ds * esz;
    m.co[0] = (uint32_t)(X + 1 < g.nx ? X + 1 : (g.xper ? 0 : X)) * esz;
    m.co[1] = (uint32_t)X * esz;
    m.co[2] = (uint32_t)(X > 0 ? X - 1 : (g.xper ? g.nx - 1 : 0)) * esz;
    m.core = inside && lane >= K - 1 && lane < K - 1 + WC && X0 + lane - (K - 1) < g.nx;
    m.outx = m.core ? (uint32_t)X * esz : ~0u;
    m.wx = inside ? (uint32_t)X * 2u : ~0u;   // dead columns: no bounce
    m.sx = (uint32_t)X * (uint32_t)sizeof(typename S::C);
    m.inlet = !g.xper && inside && X == 0;
    m.outlet = !g.xper && inside && X == g.nx - 1;
    m.has_inlet = m.any(m.inlet);
    m.has_outlet = m.any(m.outlet);
    const int half = (rows + 1) / 2;
    m.y0 = run * rows + (split && v == 1 ? half : 0);
    m.y1 = min(g.ny, split && v == 0 ? m.y0 + half : run * rows + rows);
    m.rec = rec;
    m.run();
    if constexpr (FORCE) {
        int r = 0;
        static_for<0, K>([&](auto I) {
            if ((rec >> (int)I) & 1u) {
                double fx = m.fx[I], fy = m.fy[I], fz = 0.0;
                wave_sum3(fx, fy, fz);
                if (lane == 0) {
                    double *P = partials + 3 * ((size_t)(pend + r) * nwaves + wave);
                    P[0] = fx;
                    P[1] = fy;
                    P[2] = fz;
                }
                r++;
            }
        });
    }
}

// ---- launcher of one storage format ----
template <class S>
static hipError_t strip_launch_s(const StripLaunch &l, const FusedArgs &a, hipStream_t s) {
    using T = typename S::T;
    hipError_t e = hipErrorInvalidValue;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)((l.nwaves + 3) / 4)), dim3(256), 0, s, (const T *)l.A, (T *)l.B, l.lk,
                           (const typename S::C *)l.sfrac, l.uin, l.partials, a, l.strips, l.rows, l.nwaves, l.rec, l.pend);
        e = hipGetLastError();
    };
    auto steps = [&](auto k) {
        constexpr int K = decltype(k)::value;
        if (l.steps != K) return;
        if (l.sfrac) l.rec ? go(k_strip<S, K, true, true>) : go(k_strip<S, K, false, true>);
        else l.rec ? go(k_strip<S, K, true, false>) : go(k_strip<S, K, false, false>);
    };
    steps(std::integral_constant<int, 2>{});
    steps(std::integral_constant<int, 3>{});
    steps(std::integral_constant<int, 4>{});
    return e;
}

}  // namespace lbm
