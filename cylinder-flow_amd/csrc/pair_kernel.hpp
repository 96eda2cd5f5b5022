// pair_kernel.hpp -- two D3Q27 time steps per pass over memory (plain mode, every storage format).
//
// One step moves 2Q values per node and is bound by HBM; its arithmetic takes a third to two
// thirds of that time.  k_pair therefore advances the state by two steps per launch and moves
// those 2Q values once: block b owns a WX x WY column of nodes over a run of z planes and marches
// along z.  Per plane k
//   1. every position of the column and of a one-node rim around it (TX x TY positions, one per
//      thread) pulls the first step's populations of plane k from A, with the boundary rules,
//      collides and leaves the stored values in the LDS (rounded to the storage format, so the
//      second step reads exactly what a separate launch would have read);
//   2. the threads of the column pull the second step's populations from the LDS.  Plane k holds
//      the last third (e_z < 0) of what plane k - 1 pulls, the middle third (e_z = 0) of what
//      plane k pulls and the first third (e_z > 0) of plane k + 1's, so a thread keeps 27 values
//      from plane to plane in registers and the LDS holds one plane;
//   3. plane k - 1 is complete: it collides and is stored to B.
// The loads of plane k + 1 are issued before the arithmetic of plane k and stay in flight behind
// it.  The rim is computed by every block that needs it (no block waits for another).
//
// Half-way bounce-back (walls and mask links) comes from a word per node (pair_words.hip):
// bit i, direction i takes the node's own h_opp(i).  Blocks read the words only of planes where
// the column or its rim holds one (a bit per column and plane), and only waves that hold one do
// more than the plain pull; elsewhere the pull has no rule but the x edges: the inlet's unknowns are overwritten by the inlet rule, the outlet's source is
// clamped and periodic axes wrap, all three in the lane's offsets.
//
// 512x256x256 cylinder, us per step, one step per launch / two: FP64 2525 / 1735, FP32 1197 / 875,
// FP16 630 / 572.  FP32 is bound by HBM (5.4 TB/s of L2 misses with every block in step; the rim reads
// 1.13 times the state), FP16 by instruction issue (68 % VALU busy at 309 instructions per node and
// step), FP64 by both.
//
// A recorded first step's momentum exchange is summed from the pass's input by a kernel of its own
// (pair_force_s); a second step's by the pass (FORCE): the node's own values are in the LDS when its plane's
// are pulled, three sums per node next to the mask go to memory by the node's rank (PairSeg).  Those sums
// and their stores are in every pass's straight line: 3 % of a pass in FP32 and FP64, 29 % in FP16.
//
// Every node's arithmetic is that of the one-step kernels (collide, collide_f64, velocity_inlet,
// the storage format's decode and encode), so populations and fields are theirs bit for bit.
#pragma once
#include "fast_kernel.hpp"

namespace lbm {

// Column and block of a storage format.  What bounds the choice: 27 + 27 + 27 values in registers per
// thread (in flight, in work, kept between planes) leave 3 waves per SIMD in FP32 and 16 bits, 2 in FP64;
// one plane, doubled where the 160 KB LDS hold it (DB: one barrier per plane instead of two), then
// limits the positions.  Measured on 512x256x256 (us per step): FP32 64x8 871, 64x13 in 1024 threads
// (128 registers, spilled) 888, 32x20 978; FP64 32x13 1825, 32x12 1814 (and 8 % slower on 256x128x128),
// 64x5 1920, 16x24 1925.  ROWS (see place()): FP32 871 against 921, 16 bits 644 against 576.
template <class S> struct PairTile {
    static constexpr int WX = 64, WY = 8, NT = 768;
    static constexpr bool DB = true, ROWS = sizeof(typename S::T) == 4;
};
template <> struct PairTile<SF64> {
    static constexpr int WX = 32, WY = 13, NT = 512;
    static constexpr bool DB = false, ROWS = false;
};

// rank of direction i among the directions with its e_z
constexpr int zrank(int i) {
    int k = 0;
    for (int j = 0; j < i; j++) k += Lat<27>::ez(j) == Lat<27>::ez(i);
    return k;
}

// the one-step kernels' collision of this storage format; s: sum of the populations (FP64: the
// pressure p)
template <class S, bool SFRAC>
__device__ __forceinline__ void pair_collide(const typename S::C *gv, typename S::C sf, const FusedArgs &a,
                                             typename S::C *c, typename S::C &s, typename S::C &u, typename S::C &v,
                                             typename S::C &w) {
    double fx = 0.0, fy = 0.0, fz = 0.0;
    if constexpr (sizeof(typename S::C) == 8) collide_f64<27, false, SFRAC>(gv, sf, a.tau, a.rtau, c, s, u, v, w, fx, fy, fz);
    else collide<27, false, SFRAC>(gv, sf, a.omega, c, s, u, v, w, fx, fy, fz);
}

// A plane of populations as a buffer: loads and stores take a lane offset in one VGPR and the
// direction's offset in an SGPR, and an access outside the plane is dropped by the hardware
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)bytes, 0x00027000);
}
template <class T>
__device__ __forceinline__ T buf_load(__amdgpu_buffer_rsrc_t r, uint32_t lane, uint32_t dir) {
    typename UInt<sizeof(T)>::type u;
    if constexpr (sizeof(T) == 2) u = __builtin_amdgcn_raw_buffer_load_b16(r, lane, dir, 0);
    else if constexpr (sizeof(T) == 4) u = __builtin_amdgcn_raw_buffer_load_b32(r, lane, dir, 0);
    else {
        const auto q = __builtin_amdgcn_raw_buffer_load_b64(r, lane, dir, 0);
        __builtin_memcpy(&u, &q, 8);
    }
    T v;
    __builtin_memcpy(&v, &u, sizeof(T));
    return v;
}
// (regular stores: the last-level cache keeps what the next step reads first; non-temporal ones cost
// 10 % at 453 MB per buffer in FP32, 2 % at 3.6 GB, and gain nothing in FP16 and FP64)
template <class T>
__device__ __forceinline__ void buf_store(__amdgpu_buffer_rsrc_t r, uint32_t lane, uint32_t dir, T v) {
    if constexpr (sizeof(T) == 2) {
        uint16_t u;
        __builtin_memcpy(&u, &v, 2);
        __builtin_amdgcn_raw_buffer_store_b16(u, r, lane, dir, 0);
    } else if constexpr (sizeof(T) == 4) {
        uint32_t u;
        __builtin_memcpy(&u, &v, 4);
        __builtin_amdgcn_raw_buffer_store_b32(u, r, lane, dir, 0);
    } else {
        decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0)) u;
        __builtin_memcpy(&u, &v, 8);
        __builtin_amdgcn_raw_buffer_store_b64(u, r, lane, dir, 0);
    }
}

// bit i of w ? a : b, with the bit spread over a mask (the compiler would compare and select)
__device__ __forceinline__ uint32_t pair_pick32(uint32_t m, uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}
template <class V>
__device__ __forceinline__ V pair_pick(uint32_t w, int i, V a, V b) {
    const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)w, i, 1);
    V r;
    if constexpr (sizeof(V) == 8) {
        uint32_t x[2], y[2];
        __builtin_memcpy(x, &a, 8);
        __builtin_memcpy(y, &b, 8);
        x[0] = pair_pick32(m, x[0], y[0]);
        x[1] = pair_pick32(m, x[1], y[1]);
        __builtin_memcpy(&r, x, 8);
    } else {
        typename UInt<sizeof(V)>::type x, y;
        __builtin_memcpy(&x, &a, sizeof(V));
        __builtin_memcpy(&y, &b, sizeof(V));
        x = (decltype(x))pair_pick32(m, x, y);
        __builtin_memcpy(&r, &x, sizeof(V));
    }
    return r;
}

// LDS of a block: one plane of stored values, then the column's own bounced values (see k_pair)
template <class S>
constexpr size_t pair_lds_bytes() {
    using P = PairTile<S>;
    return sizeof(typename S::T) * ((P::DB ? 2 : 1) * 27 * (P::WX + 2) * (P::WY + 2) + 9 * P::WX * P::WY);
}

// the value in a register of its own, formed here (so that the register it came from can take the
// next load)
template <class C>
__device__ __forceinline__ C pinned(C v) {
    if constexpr (sizeof(C) == 4) {
        C r;
        asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
        return r;
    } else {
        uint32_t u[2], r[2];
        __builtin_memcpy(u, &v, 8);
        asm volatile("v_mov_b32 %0, %2\n\tv_mov_b32 %1, %3" : "=&v"(r[0]), "=&v"(r[1]) : "v"(u[0]), "v"(u[1]));
        C o;
        __builtin_memcpy(&o, r, 8);
        return o;
    }
}

// The march of one block.  A pass k takes plane k from the LDS for the second step and puts plane k + 1 of the first step
// into it.  The passes are straight-line code in all that touches global memory: a branch around a
// load or store would make the wait for plane k + 1's loads wait for the stores behind them as well.
template <class S, bool SFRAC, bool MACROS, bool FORCE>
struct PairMarch {
    using L = Lat<27>;
    using T = typename S::T;
    using C = typename S::C;
    using P = PairTile<S>;
    static constexpr int Q = 27, WX = P::WX, WY = P::WY, TX = WX + 2, TY = WY + 2, NP = TX * TY;
    static constexpr bool DB = P::DB;
    // At the inlet the nodes x = 0 run a long sequence of their own: the first step's go to the
    // threads from IN1 on (a wave of their own where there is room), the second step's to the last
    // wave, so that each costs one wave and not every wave of the block.
    static constexpr int IN1 = (TY * WX + 63) / 64 * 64 + 2 * TY <= P::NT ? (TY * WX + 63) / 64 * 64 : TY * WX, IN2 = P::NT - 64;
    static_assert(NP <= P::NT && WX * WY <= P::NT, "one thread per position and per node of the column");
    static_assert(IN1 + 2 * TY <= P::NT && WX * WY <= IN2 && WY <= 64, "inlet threads");
    typedef const __attribute__((address_space(4))) uint32_t *cword;   // constant: scalar loads

    const T *A;
    T *B;
    const uint32_t *bw;
    const C *sfrac;
    const double *uin;
    double *macros;
    // FORCE: the second step's momentum exchange, three doubles per node next to the mask, in node order
    const PairSeg *seg;
    double *trip;
    uint32_t tripb;   // bytes of trip
    const FusedArgs &a;
    T *lds;
    cword tf;   // bit k of the column's words: plane k holds a bounce word
    int z0, z1;
    uint32_t planeb, planen, dsb;
    // this thread's position (first step) and node (second step)
    bool act1, act2, inl1, inl2;
    bool first, second;   // whether any thread of the wave has one
    int idx1, i0, iP, iM, y1, y2;
    uint32_t node1, node2, out2, ro[3], co[3];
    T *ownv;
    // raw populations of the next plane (in flight), inlet velocity, solid fraction and bounce words
    T R[Q];
    double u1, u2;
    C sf1, sf2;
    uint32_t w1, w2, w2k;
    uint32_t wally;                    // FORCE: the directions that cross a y wall
    uint32_t sbase, slo, shi;          // and the segment of the next pass's plane
    T upJ[9], midJ[9], upK[9];   // pulled values of plane k - 1 (e_z > 0, e_z = 0) and of plane k (e_z > 0)

    // bounce word of a node of plane k: 0 without a memory access where the plane holds none (the
    // buffer is empty then)
    __device__ __forceinline__ uint32_t word(int k, uint32_t node) const {
        const uint32_t on = (tf[k >> 5] >> (k & 31)) & 1u;
        return buf_load<uint32_t>(plane_rsrc(bw + (size_t)planen * k, on * planen * 4u), node * 4u, 0);
    }
    template <class F>
    static constexpr uint32_t dirs(F f) {
        uint32_t b = 0;
        for (int i = 1; i < Q; i++)
            if (f(i)) b |= 1u << i;
        return b;
    }
    // whether any lane of the wave holds one of these bits
    __device__ __forceinline__ static bool any(uint32_t bits) { return __builtin_amdgcn_ballot_w64(bits != 0u) != 0ull; }
    // planes beyond a wall: the wall's own plane (what is pulled from it is replaced by the bounce)
    __device__ __forceinline__ int wrapz(int k) const {
        const int n = a.g.nz;
        const int clamped = min(max(k, 0), n - 1), wrapped = k + (k < 0 ? n : 0) - (k >= n ? n : 0);
        return __builtin_amdgcn_readfirstlane(a.g.zper ? max(wrapped, 0) : clamped);
    }

    __device__ __forceinline__ void place(int X0, int Y0) {
        const Geo &g = a.g;
        const int t = (int)threadIdx.x;
        // Threads to positions.  ROWS: the column's own x range row by row, so that a wave's rows start
        // on cache lines, then the rim's two side columns; otherwise every position, x fastest.  At the
        // inlet the left side column lies outside; the nodes x = 0 go to the threads from IN1 on.
        const bool inl_tile = !g.xper && X0 == 0;
        int px, py;
        if constexpr (P::ROWS) {
            const int e = t - IN1;
            const bool side = t >= IN1 && e < 2 * TY;
            px = side ? (e >= TY ? TX - 1 : (inl_tile ? 1 : 0)) : 1 + t % WX;
            py = side ? e % TY : t / WX;
            act1 = side || (t < TY * WX && !(inl_tile && px == 1));
        } else if (!inl_tile) {
            px = t % TX;
            py = t / TX;
            act1 = t < NP;
        } else {
            px = t < TY * WX ? 2 + t % WX : 1;
            py = t < TY * WX ? t / WX : t - IN1;
            act1 = t < TY * WX || (t >= IN1 && t < IN1 + TY);
        }
        const bool last_wave = inl_tile && t >= IN2 && t < IN2 + WY;
        const int cx = last_wave ? 0 : t % WX, cy = last_wave ? t - IN2 : t / WX;
        act2 = last_wave || (t < WX * WY && !(inl_tile && cx == 0));
        first = any(act1);
        second = any(act2);
        // first step: node, sources; positions outside the domain load from node (0, 0)
        int X = X0 - 1 + px, Y = Y0 - 1 + py;
        if (g.xper) X = X < 0 ? X + g.nx : (X >= g.nx ? X - g.nx : X);
        if (g.yper) Y = Y < 0 ? Y + g.ny : (Y >= g.ny ? Y - g.ny : Y);
        act1 = act1 && X >= 0 && X < g.nx && Y >= 0 && Y < g.ny;
        if (!act1) X = Y = 0;
        inl1 = inl_tile && act1 && X == 0;
        idx1 = py * TX + px;
        y1 = Y;
        planen = (uint32_t)g.nxp * (uint32_t)g.ny;              // nodes of a plane (padded)
        node1 = (uint32_t)X + (uint32_t)g.nxp * (uint32_t)Y;    // within its plane
        // byte offsets of the sources within their plane's rows: row e_y = -1, 0, +1 (y + 1, y, y - 1)
        // and column e_x = -1, 0, +1
        const uint32_t rsb = (uint32_t)(g.rs * sizeof(T)), esz = (uint32_t)sizeof(T);
        ro[0] = (uint32_t)(Y + 1 < g.ny ? Y + 1 : (g.yper ? 0 : Y)) * rsb;
        ro[1] = (uint32_t)Y * rsb;
        ro[2] = (uint32_t)(Y > 0 ? Y - 1 : (g.yper ? g.ny - 1 : 0)) * rsb;
        co[0] = (uint32_t)(X + 1 < g.nx ? X + 1 : (g.xper ? 0 : X)) * esz;
        co[1] = (uint32_t)X * esz;
        co[2] = (uint32_t)(X > 0 ? X - 1 : (g.xper ? g.nx - 1 : 0)) * esz;
        // second step: node, LDS positions (e_x = +1, 0, -1; the outlet's source clamped); a lane
        // beyond the domain stores outside its buffer, which the hardware drops
        const int X2 = X0 + cx, Y2 = Y0 + cy;
        act2 = act2 && X2 < g.nx && Y2 < g.ny;
        inl2 = inl_tile && act2 && X2 == 0;
        i0 = act2 ? (cy + 1) * TX + cx + 1 : TX + 1;
        iP = i0 - 1;
        iM = (!g.xper && X2 == g.nx - 1) ? i0 : i0 + 1;
        y2 = act2 ? Y2 : 0;
        node2 = act2 ? (uint32_t)X2 + (uint32_t)g.nxp * (uint32_t)Y2 : 0u;
        out2 = act2 ? (uint32_t)Y2 * rsb + (uint32_t)X2 * esz : ~0u;
        ownv = lds + (DB ? 2 : 1) * Q * NP + (act2 ? cy * WX + cx : 0);   // its node's 9 slots, WX * WY apart
        if constexpr (FORCE) {
            wally = 0u;
            if (!g.yper && Y2 == 0) wally |= dirs([](int i) { return L::ey(i) > 0; });
            if (!g.yper && Y2 == g.ny - 1) wally |= dirs([](int i) { return L::ey(i) < 0; });
        }
        sbase = slo = shi = 0;
        planeb = (uint32_t)(g.rs * (size_t)g.ny * sizeof(T));
        dsb = (uint32_t)(g.ds * sizeof(T));
        static_for<0, Q>([&](auto I) { R[I] = T(0); });
        static_for<0, 9>([&](auto I) { upJ[I] = midJ[I] = upK[I] = T(0); });
        u1 = u2 = 0.0;
        sf1 = sf2 = 0;
        w1 = w2 = w2k = 0;
    }

    // Issues the loads of plane k: the planes k - 1, k, k + 1 as one buffer from the lowest of them
    // (periodic z wraps: up to the whole state, which the host keeps below 4 GiB); a direction's row
    // starts at a scalar offset, a bounced lane (word w1, loaded one pass before) takes its own
    // row's opposite direction instead.  With them what pass `pass` + 1's second step needs.
    template <bool FIRST, bool SECOND>
    __device__ __forceinline__ void issue(int k, int pass) {
        const int kk = wrapz(k), km = wrapz(kk - 1), kp = wrapz(kk + 1);
        const int lo = __builtin_amdgcn_readfirstlane(min(kk, min(km, kp)));
        const int hi = __builtin_amdgcn_readfirstlane(max(kk, max(km, kp)));
        const auto rs = plane_rsrc((const char *)A + (size_t)planeb * lo, planeb * (uint32_t)(hi - lo + 1));
        const uint32_t s0 = planeb * (uint32_t)(kk - lo), sm = planeb * (uint32_t)(km - lo), sp = planeb * (uint32_t)(kp - lo);
        const int j = wrapz(pass);   // the plane the next pass's second step completes
        if (FIRST && inl1) u1 = uin[y1 + a.g.ny * kk];
        if (SECOND && inl2) u2 = uin[y2 + a.g.ny * j];
        if constexpr (SFRAC && FIRST) sf1 = sfrac[node1 + (size_t)planen * kk];
        if constexpr (SFRAC && SECOND) sf2 = sfrac[node2 + (size_t)planen * j];
        if constexpr (SECOND) w2k = word(wrapz(pass + 1), node2);   // of the next pass's plane
        if constexpr (FORCE && SECOND) {
            const int n = wrapz(pass + 1);
            const uint32_t on = (tf[n >> 5] >> (n & 31)) & 1u, segs = planen >> 6;
            const auto rs = plane_rsrc(seg + (size_t)segs * n, on * segs * (uint32_t)sizeof(PairSeg));
            const uint32_t at = (node2 >> 6) * (uint32_t)sizeof(PairSeg);
            sbase = buf_load<uint32_t>(rs, at, 0);
            slo = buf_load<uint32_t>(rs, at, 4);
            shi = buf_load<uint32_t>(rs, at, 8);
        }
        if constexpr (FIRST) {
            const uint32_t w = w1;
            w1 = word(wrapz(k + 1), node1);
            // opaque, so that the nine sums below are formed here and not kept in registers
            uint32_t rr[3] = {ro[0], ro[1], ro[2]};
            asm volatile("" : "+v"(rr[0]), "+v"(rr[1]), "+v"(rr[2]));
            if (any(w)) {
                const uint32_t here = rr[1] + co[1];
                static_for<0, Q>([&](auto I) {
                    constexpr int i = I;
                    const uint32_t nom = rr[L::ey(i) + 1] + co[L::ex(i) + 1] + ((L::ez(i) > 0 ? sm : L::ez(i) < 0 ? sp : s0) + i * dsb);
                    const uint32_t own = here + (s0 + L::opp(i) * dsb);
                    R[i] = buf_load<T>(rs, pair_pick<uint32_t>(w, i, own, nom), 0);
                });
            } else {
                static_for<0, Q>([&](auto I) {
                    constexpr int i = I;
                    R[i] = buf_load<T>(rs, rr[L::ey(i) + 1] + co[L::ex(i) + 1], (L::ez(i) > 0 ? sm : L::ez(i) < 0 ? sp : s0) + i * dsb);
                });
            }
        }
    }

    // the LDS slot direction I is pulled from
    template <int i>
    __device__ __forceinline__ int at() const {
        return i * NP + (L::ex(i) > 0 ? iP : L::ex(i) < 0 ? iM : i0) - L::ey(i) * TX;
    }

    // the second step of plane j = k - 1, completed by plane k in `in`
    __device__ __forceinline__ void complete(int j, const T *in) {
        T r[Q];
        static_for<0, Q>([&](auto I) {
            constexpr int i = I;
            if constexpr (L::ez(i) > 0) r[i] = upJ[zrank(i)];
            else if constexpr (L::ez(i) == 0) r[i] = midJ[zrank(i)];
            else r[i] = in[at<i>()];
        });
        if (any(w2))
            static_for<1, Q>([&](auto I) {
                constexpr int i = I;
                if constexpr (L::ez(i) < 0) {
                    const T o = ownv[zrank(i) * WX * WY];
                    r[i] = pair_pick<T>(w2, i, o, r[i]);
                }
            });
        C g[Q], c[Q], s, u, v, w;
        static_for<0, Q>([&](auto I) { g[I] = S::template decode<I, L>(r[I], 0.f); });
        if (inl2) velocity_inlet<Q, C>(g, (C)u2);
        pair_collide<S, SFRAC>(g, sf2, a, c, s, u, v, w);
        const auto rs = plane_rsrc((char *)B + (size_t)planeb * j, planeb);
        static_for<0, Q>([&](auto I) { buf_store<T>(rs, out2, (uint32_t)I * dsb, S::template enc<I, L>(c[I], StoreParams{})); });
        if constexpr (MACROS)
            if (act2) {
                double *m = macros + node2 + (size_t)planen * j;
                m[0] = sizeof(C) == 8 ? (double)s : (double)s * (1.0 / 3.0);
                m[a.g.plane] = (double)u;
                m[2 * a.g.plane] = (double)v;
                m[3 * a.g.plane] = (double)w;
            }
    }

    // plane k's middle third, plane k + 1's first third; plane k's bounced directions (those along
    // e_z < 0 kept in the LDS for the next pass: they are complete with plane k + 1)
    __device__ __forceinline__ void collect(int k, const T *in) {
        static_for<0, 9>([&](auto I) { upJ[I] = upK[I]; });
        static_for<0, Q>([&](auto I) {
            constexpr int i = I;
            if constexpr (L::ez(i) == 0) midJ[zrank(i)] = in[at<i>()];
            else if constexpr (L::ez(i) > 0) upK[zrank(i)] = in[at<i>()];
        });
        w2 = w2k;
        if (any(w2))
            static_for<1, Q>([&](auto I) {
                constexpr int i = I;
                const T o = in[L::opp(i) * NP + i0];
                if constexpr (L::ez(i) == 0) midJ[zrank(i)] = pair_pick<T>(w2, i, o, midJ[zrank(i)]);
                else if constexpr (L::ez(i) > 0) upJ[zrank(i)] = pair_pick<T>(w2, i, o, upJ[zrank(i)]);
                else if (act2) ownv[zrank(i) * WX * WY] = o;
            });
        if constexpr (FORCE) {
            // the mask's links of plane k from the node's own values (all of them are in the LDS now), in
            // direction order; a store that the buffer drops where there are none
            double f[3] = {0.0, 0.0, 0.0};
            uint32_t wall = wally;
            if (!a.g.zper && k == 0) wall |= dirs([](int i) { return L::ez(i) > 0; });
            if (!a.g.zper && k == a.g.nz - 1) wall |= dirs([](int i) { return L::ez(i) < 0; });
            const uint32_t links = w2 & ~wall;
            uint32_t dst = ~0u;
            if (any(links)) {
                static_for<1, Q>([&](auto I) {
                    constexpr int i = I;
                    constexpr int ex = L::ex(i), ey = L::ey(i), ez = L::ez(i);
                    const double m = 2.0 * (double)S::template decode<i, L>(in[L::opp(i) * NP + i0], 0.f);
                    const bool on = (links >> i) & 1u;
                    if constexpr (ex != 0) f[0] = on ? f[0] - ex * m : f[0];
                    if constexpr (ey != 0) f[1] = on ? f[1] - ey * m : f[1];
                    if constexpr (ez != 0) f[2] = on ? f[2] - ez * m : f[2];
                });
            }
            const uint32_t bit = node2 & 63u;
            const unsigned long long held = (unsigned long long)slo | (unsigned long long)shi << 32;
            // (a node next to the mask whose links are all clamped away or inlet unknowns stores its zeros)
            if (act2 && k >= z0 && k < z1 && ((held >> bit) & 1ull))
                dst = (sbase + (uint32_t)__builtin_popcountll(held & ((1ull << bit) - 1ull))) * 24u;
            const auto rs = plane_rsrc(trip, tripb);
            static_for<0, 3>([&](auto D) { buf_store<double>(rs, dst, (uint32_t)D * 8u, f[D]); });
        }
    }

    // passes lo .. hi of a wave with positions of the first step (FIRST), with nodes of the column
    // (COLLECT), and whether plane k - 1 is one of the block's (SECOND)
    template <bool FIRST, bool COLLECT, bool SECOND>
    __device__ __forceinline__ void passes(int lo, int hi) {
        for (int k = lo; k <= hi; k++) {
            const T *const in = lds + (DB ? (k & 1) * Q * NP : 0);
            T *const next = lds + (DB ? (~k & 1) * Q * NP : 0);
            if constexpr (SECOND) complete(k - 1, in);
            if (k == z1) break;
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (COLLECT) collect(k, in);
            C g[Q], c[Q], s, u, v, w;
            if constexpr (FIRST) static_for<0, Q>([&](auto I) { g[I] = pinned<C>(S::template decode<I, L>(R[I], 0.f)); });
            const double uc = u1;
            const C sc = sf1;
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (FIRST || COLLECT) issue<FIRST, COLLECT>(k + 2 <= z1 ? k + 2 : z1, k);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (FIRST) {
                if (inl1) velocity_inlet<Q, C>(g, (C)uc);
                pair_collide<S, SFRAC>(g, sc, a, c, s, u, v, w);
            }
            if constexpr (!DB) lds_barrier();   // one buffer: plane k is read
            if constexpr (FIRST)
                if (act1) static_for<0, Q>([&](auto I) { next[I * NP + idx1] = S::template enc<I, L>(c[I], StoreParams{}); });
            lds_barrier();
        }
    }

    __device__ __forceinline__ void run() {
        if (first) w1 = word(wrapz(z0 - 1), node1);
        // plane z0 - 1 is the first one needed; pass z0 + 1 completes plane z0
        if (first) issue<true, false>(z0 - 1, z0 - 3);
        if (first && second) {
            passes<true, true, false>(z0 - 2, z0);
            passes<true, true, true>(z0 + 1, z1);
        } else if (first) {
            passes<true, false, false>(z0 - 2, z1);
        } else if (second) {
            passes<false, true, false>(z0 - 2, z0);
            passes<false, true, true>(z0 + 1, z1);
        } else {
            passes<false, false, false>(z0 - 2, z1);
        }
    }
};

template <class S, bool SFRAC, bool MACROS, bool FORCE>
__global__ void __launch_bounds__(PairTile<S>::NT)
    k_pair(const typename S::T *__restrict__ A, typename S::T *__restrict__ B, const uint32_t *__restrict__ bw,
           const uint32_t *__restrict__ tflag, const typename S::C *__restrict__ sfrac, const double *__restrict__ uin,
           double *__restrict__ macros, const PairSeg *__restrict__ seg, double *__restrict__ trip, uint32_t tripb, const FusedArgs a,
           int tiles_x, int tiles_y, int cz) {
    extern __shared__ __align__(16) char pair_lds[];
    using T = typename S::T;
    const Geo &g = a.g;
    // workgroups go to the 8 XCDs in turn: XCD x takes a run of neighbouring columns, whose rims
    // then meet in one L2
    const int n = (int)gridDim.x, xcd = (int)(blockIdx.x % 8u);
    const int pos = xcd * (n / 8) + min(xcd, n % 8) + (int)(blockIdx.x / 8u);
    // (the quotients are uniform; readfirstlane keeps what follows from them in scalar registers)
    const int tiles = tiles_x * tiles_y, chunk = __builtin_amdgcn_readfirstlane(pos / tiles), tile = pos - chunk * tiles;
    const int ty = __builtin_amdgcn_readfirstlane(tile / tiles_x);
    const int z0 = chunk * cz, z1 = min(g.nz, z0 + cz);
    PairMarch<S, SFRAC, MACROS, FORCE> m{A, B, bw, sfrac, uin, macros, seg, trip, tripb, a};
    typedef typename PairMarch<S, SFRAC, MACROS, FORCE>::cword cword;
    m.lds = (T *)pair_lds;
    m.tf = (cword)(uintptr_t)(tflag + (size_t)tile * ((g.nz + 31) / 32));
    m.z0 = z0;
    m.z1 = z1;
    m.place((tile - ty * tiles_x) * PairTile<S>::WX, ty * PairTile<S>::WY);
    m.run();
}

// Momentum exchange of the mask links per block of a row, block b (list[b] = its index along the rows)
// into slot b, from a step's input: each node's links summed in direction order and the nodes of a
// block as the one-step kernels with per-block slots do it (k_fused, k_dense_v), bit for bit.
template <class S>
__global__ void __launch_bounds__(256)
    k_block_force(const typename S::T *__restrict__ A, const uint32_t *__restrict__ bw, const uint32_t *__restrict__ list, int gx,
                  double *__restrict__ partials, const FusedArgs a) {
    using L = Lat<27>;
    constexpr int Q = 27;
    const Geo &g = a.g;
    const uint32_t id = list[blockIdx.x], row = id / (uint32_t)gx;
    const uint32_t x = (id - row * (uint32_t)gx) * blockDim.x + threadIdx.x;
    const int y = (int)(row % (uint32_t)g.ny), z = (int)(row / (uint32_t)g.ny);
    uint32_t lk = x < (uint32_t)g.nx ? bw[x + (size_t)g.nxp * row] : 0u;
    static_for<1, Q>([&](auto I) {   // walls bounce without force
        constexpr int i = I;
        const int sy = y - L::ey(i), sz = z - L::ez(i);
        if ((!g.yper && (unsigned)sy >= (unsigned)g.ny) || (!g.zper && (unsigned)sz >= (unsigned)g.nz)) lk &= ~(1u << i);
    });
    double fx = 0.0, fy = 0.0, fz = 0.0;
    if (lk != 0u) {
        typename S::T val[Q];
        static_for<1, Q>([&](auto I) {   // all loads first; a direction without a link loads its rest value
            constexpr int i = I;
            val[i] = A[pel(g, ((lk >> i) & 1u) ? L::opp(i) : 0, x, row)];
        });
        static_for<1, Q>([&](auto I) {
            constexpr int i = I;
            constexpr int ex = L::ex(i), ey = L::ey(i), ez = L::ez(i), o = L::opp(i);
            if ((lk >> i) & 1u) {
                const double m = 2.0 * (double)S::template decode<i, L>(val[i], a.sp.off[o]);
                if constexpr (ex != 0) fx -= ex * m;
                if constexpr (ey != 0) fy -= ey * m;
                if constexpr (ez != 0) fz -= ez * m;
            }
        });
    }
    __shared__ double red[3 * 4];
    block_sum3<4>(fx, fy, fz, red);
    if (threadIdx.x == 0) {
        partials[3 * (size_t)blockIdx.x] = fx;
        partials[3 * (size_t)blockIdx.x + 1] = fy;
        partials[3 * (size_t)blockIdx.x + 2] = fz;
    }
}

// The same per-block sums from the nodes' own (k_pair, FORCE).
template <class S>
__global__ void __launch_bounds__(256)
    k_block_sum(const PairSeg *__restrict__ seg, const double *__restrict__ trip, const uint32_t *__restrict__ list, int gx,
                double *__restrict__ partials, Geo g) {
    const uint32_t id = list[blockIdx.x], row = id / (uint32_t)gx;
    const uint32_t x = (id - row * (uint32_t)gx) * blockDim.x + threadIdx.x;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    if (x < (uint32_t)g.nx) {
        const PairSeg q = seg[(x + (size_t)g.nxp * row) >> 6];
        const unsigned long long held = (unsigned long long)q.lo | (unsigned long long)q.hi << 32;
        const uint32_t bit = x & 63u;
        if ((held >> bit) & 1ull) {
            const double *t = trip + 3 * (size_t)(q.base + (uint32_t)__builtin_popcountll(held & ((1ull << bit) - 1ull)));
            fx = t[0];
            fy = t[1];
            fz = t[2];
        }
    }
    __shared__ double red[3 * 4];
    block_sum3<4>(fx, fy, fz, red);
    if (threadIdx.x == 0) {
        partials[3 * (size_t)blockIdx.x] = fx;
        partials[3 * (size_t)blockIdx.x + 1] = fy;
        partials[3 * (size_t)blockIdx.x + 2] = fz;
    }
}

// ---- launchers of one storage format (pair_f64.hip ... pair_bf16.hip) ----
template <class S>
static hipError_t pair_prepare_s() {
    const int bytes = (int)pair_lds_bytes<S>();
    for (const void *k : {(const void *)k_pair<S, false, false, false>, (const void *)k_pair<S, false, true, false>,
                          (const void *)k_pair<S, true, false, false>, (const void *)k_pair<S, true, true, false>,
                          (const void *)k_pair<S, false, false, true>}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <class S>
static hipError_t pair_step_s(const PairPlan &p, const void *A, void *B, const void *sfrac, const double *uin,
                              double *macros, bool mac, double *trip, const FusedArgs &a, hipStream_t s) {
    using T = typename S::T;
    using C = typename S::C;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles_x * p.tiles_y * p.chunks)), dim3(PairTile<S>::NT),
                           (unsigned)pair_lds_bytes<S>(), s, (const T *)A, (T *)B, p.bw, p.tflag, (const C *)sfrac, uin,
                           macros, p.seg, trip, (uint32_t)(24u * (uint32_t)p.nnear), a, p.tiles_x, p.tiles_y, p.cz);
    };
    if (trip) {
        if (sfrac || mac) return hipErrorInvalidValue;
        go(k_pair<S, false, false, true>);
    } else if (sfrac) mac ? go(k_pair<S, true, true, false>) : go(k_pair<S, true, false, false>);
    else mac ? go(k_pair<S, false, true, false>) : go(k_pair<S, false, false, false>);
    return hipGetLastError();
}

// the momentum exchange of the first of the two steps, from its input (k_link_force, k_block_force)
template <class S>
static hipError_t pair_force_s(const PairPlan &p, const void *A, double *partials, const FusedArgs &a, hipStream_t s) {
    if (p.nslots == 0) return hipSuccess;
    if (p.fblk) {
        hipLaunchKernelGGL(k_block_force<S>, dim3((unsigned)p.nslots), dim3(p.fbx), 0, s, (const typename S::T *)A, p.bw, p.fblk,
                           p.fgx, partials, a);
        return hipGetLastError();
    }
    hipLaunchKernelGGL((k_link_force<27, S>), dim3((unsigned)((p.nlink + 255) / 256)), dim3(256), 0, s,
                       (const typename S::T *)A, p.link, p.linklk, p.link_slot, p.nlink, partials, a);
    return hipGetLastError();
}

// after a pair whose second step records the force, with per-block slots: p.trip into partials
template <class S>
static hipError_t pair_block_sum_s(const PairPlan &p, double *partials, const FusedArgs &a, hipStream_t s) {
    if (p.nslots == 0) return hipSuccess;
    hipLaunchKernelGGL(k_block_sum<S>, dim3((unsigned)p.nslots), dim3(p.fbx), 0, s, p.seg, p.trip, p.fblk, p.fgx, partials, a.g);
    return hipGetLastError();
}

template <class S>
constexpr PairOps pair_ops() {
    return {PairTile<S>::WX, PairTile<S>::WY, pair_lds_bytes<S>(), pair_prepare_s<S>, pair_step_s<S>, pair_force_s<S>, pair_block_sum_s<S>};
}

}  // namespace lbm
