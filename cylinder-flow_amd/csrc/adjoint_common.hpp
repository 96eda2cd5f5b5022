// adjoint_common.hpp -- one reverse step of a node, shared by the adjoint kernels (adjoint_kernels.hip,
// adjoint_small.hip).
#pragma once
#include "fused_common.hpp"

namespace lbm {

// a*b + c rounded once (FP32 or FP64)
template <class C>
__device__ __forceinline__ C fmac(C a, C b, C c) {
    if constexpr (sizeof(C) == 4) return __builtin_fmaf(a, b, c);
    else return __builtin_fma(a, b, c);
}

// e_i . u with the zero components of e_i skipped
template <class L, int i, class C>
__device__ __forceinline__ C edot(const C *u) {
    C r = 0;
    bool first = true;
    static_for<0, 3>([&](auto K) {
        constexpr int k = K;
        constexpr int e = k == 0 ? L::ex(i) : (k == 1 ? L::ey(i) : L::ez(i));
        if constexpr (e != 0) {
            const C t = e > 0 ? u[k] : -u[k];
            r = first ? t : r + t;
            first = false;
        }
    });
    return r;
}

// Transposes of the inlet's regularisation and Zou-He completion applied to m = mu_m at an inlet
// node (x = 0, x not periodic), in place, and their contribution to dJ/du_in of its row.
template <int Q, class S>
__device__ __forceinline__ void adj_inlet_transpose(typename S::C *m, double &du) {
    using L = Lat<Q>;
    using C = typename S::C;
    // regularisation g_i = w_i (S + 3 e_ix U + 4.5 Q_i:P) is g -> A g + 3 w e_x U with
    // A_ij = w_i (1 + 4.5 Q_i:Q_j), so (A^T m)_j = M0 + 4.5 Q_j:T, M0 = sum w_i m_i,
    // T = sum w_i m_i Q_i (same structure as the forward with S -> M0, P -> T)
    {
        C M0 = 0, Rxx = 0, Ryy = 0, Rzz = 0, Rxy = 0, Rxz = 0, Ryz = 0;
        static_for<0, Q>([&](auto I) {
            constexpr int i = I;
            constexpr int ex = L::ex(i), ey = L::ey(i), ez = L::ez(i);
            const C wm = (C)L::w(i) * m[i];
            M0 += wm;
            if constexpr (ex != 0) Rxx += wm;
            if constexpr (ey != 0) Ryy += wm;
            if constexpr (ez != 0) Rzz += wm;
            if constexpr (ex * ey != 0) Rxy += (C)(ex * ey) * wm;
            if constexpr (ex * ez != 0) Rxz += (C)(ex * ez) * wm;
            if constexpr (ey * ez != 0) Ryz += (C)(ey * ez) * wm;
            if constexpr (ex != 0) du += (double)wm * (3.0 * ex);
        });
        const C M3 = M0 * (C)(1.0 / 3.0);
        const C Txx = Rxx - M3, Tyy = Ryy - M3, Tzz = Rzz - M3;
        const C d = (L::D == 3 ? Txx + Tyy + Tzz : Txx + Tyy) * (C)(1.0 / 3.0);
        static_for<0, Q>([&](auto J) {
            constexpr int j = J;
            constexpr int ex = L::ex(j), ey = L::ey(j), ez = L::ez(j);
            C q = -d, o = 0;
            if constexpr (ex != 0) q += Txx;
            if constexpr (ey != 0) q += Tyy;
            if constexpr (ez != 0) q += Tzz;
            if constexpr (ex * ey != 0) o += (C)(ex * ey) * Rxy;
            if constexpr (ex * ez != 0) o += (C)(ex * ez) * Rxz;
            if constexpr (ey * ez != 0) o += (C)(ey * ez) * Ryz;
            m[j] = M0 + ((C)4.5 * q + (C)9 * o);
        });
    }
    // Zou-He g_i = g_opp(i) + 6 w_i U - 18 w_i (e_iy N_y + e_iz N_z), N_t = sum_{e_kx=0} g_k e_kt
    static_for<0, Q>([&](auto I) {
        constexpr int i = I;
        if constexpr (L::ex(i) > 0) {
            const C mi = m[i];
            m[L::opp(i)] += mi;
            static_for<0, Q>([&](auto K) {
                constexpr int k = K;
                constexpr int dot = L::ey(i) * L::ey(k) + L::ez(i) * L::ez(k);
                if constexpr (L::ex(k) == 0 && dot != 0) m[k] += mi * (C)(-18.0 * L::w(i) * dot);
            });
            du += (double)mi * (6.0 * L::w(i));
            m[i] = 0;
        }
    });
}

// index of the direction with components (ex, ey, ez)
template <class L>
__host__ __device__ constexpr int dir_of(int ex, int ey, int ez) {
    for (int i = 0; i < (L::D == 3 ? 27 : 9); i++)
        if (L::ex(i) == ex && L::ey(i) == ey && L::ez(i) == ez) return i;
    return -1;
}

// Sums over the lattice taken one axis at a time: a line of three values v(-1), v(0), v(+1)
// along an axis becomes v(+1) + v(-1) + c v(0) (the sum, with the weight ratio c), v(+1) - v(-1)
// (first moment) and v(+1) + v(-1) (second moment).
//
// moments01: rho = sum g, j = sum g e (c = 1).
template <class L, class C>
__device__ __forceinline__ void moments01(const C *g, C &rho, C *j) {
    constexpr int NZ = L::D == 3 ? 3 : 1;
    C a0[3], a1[3], b0[3];
    static_for<0, NZ>([&](auto ZZ) {
        constexpr int ez = L::D == 3 ? (int)ZZ - 1 : 0;
        C s0[3], s1[3];
        static_for<0, 3>([&](auto YY) {
            constexpr int ey = (int)YY - 1;
            const C fp = g[dir_of<L>(1, ey, ez)], fm = g[dir_of<L>(-1, ey, ez)];
            s0[YY] = (fp + fm) + g[dir_of<L>(0, ey, ez)];
            s1[YY] = fp - fm;
        });
        a0[ZZ] = (s0[2] + s0[0]) + s0[1];
        a1[ZZ] = s0[2] - s0[0];
        b0[ZZ] = (s1[2] + s1[0]) + s1[1];
    });
    if constexpr (L::D == 3) {
        rho = (a0[2] + a0[0]) + a0[1];
        j[0] = (b0[2] + b0[0]) + b0[1];
        j[1] = (a1[2] + a1[0]) + a1[1];
        j[2] = a0[2] - a0[0];
    } else {
        rho = a0[0];
        j[0] = b0[0];
        j[1] = a1[0];
        j[2] = 0;
    }
}

// the product form of the weights that wmoments relies on
template <class L>
constexpr bool weights_factor() {
    for (int i = 0; i < (L::D == 3 ? 27 : 9); i++) {
        double p = 1.0;
        const int e[3] = {L::ex(i), L::ey(i), L::ez(i)};
        for (int a = 0; a < L::D; a++) p *= e[a] == 0 ? 4.0 / 6.0 : 1.0 / 6.0;
        const double d = p - L::w(i);
        if (d > 1e-15 || d < -1e-15) return false;
    }
    return true;
}
static_assert(weights_factor<Lat<9>>() && weights_factor<Lat<27>>(), "lattice weights are products over the axes");

// wmoments: moments of w_i f_i to second order, M0 = sum w f, M1 = sum w f e, M2 = sum w f e e^T
// as (xx, yy, zz, xy, xz, yz).  The weights are products over the axes, w(e) = prod_a w1(e_a) with
// w1(0) = 4/6 and w1(+-1) = 1/6, so each axis pass uses c = 4 and the factor 6^-D comes last.
template <class L, class C>
__device__ __forceinline__ void wmoments(const C *f, C &M0, C *M1, C *M2) {
    constexpr int NZ = L::D == 3 ? 3 : 1;
    C a0[3], a1[3], a2[3], b0[3], b1[3], c0[3];
    static_for<0, NZ>([&](auto ZZ) {
        constexpr int ez = L::D == 3 ? (int)ZZ - 1 : 0;
        C s0[3], s1[3], s2[3];
        static_for<0, 3>([&](auto YY) {
            constexpr int ey = (int)YY - 1;
            const C fp = f[dir_of<L>(1, ey, ez)], fm = f[dir_of<L>(-1, ey, ez)];
            const C t = fp + fm;
            s0[YY] = fmac((C)4, f[dir_of<L>(0, ey, ez)], t);
            s1[YY] = fp - fm;
            s2[YY] = t;
        });
        const C t0 = s0[2] + s0[0], t1 = s1[2] + s1[0];
        a0[ZZ] = fmac((C)4, s0[1], t0);
        a1[ZZ] = s0[2] - s0[0];
        a2[ZZ] = t0;
        b0[ZZ] = fmac((C)4, s1[1], t1);
        b1[ZZ] = s1[2] - s1[0];
        c0[ZZ] = fmac((C)4, s2[1], s2[2] + s2[0]);
    });
    C r[10];
    if constexpr (L::D == 3) {
        const C t = a0[2] + a0[0];
        r[0] = fmac((C)4, a0[1], t);                    // M0
        r[1] = fmac((C)4, b0[1], b0[2] + b0[0]);        // x
        r[2] = fmac((C)4, a1[1], a1[2] + a1[0]);        // y
        r[3] = a0[2] - a0[0];                           // z
        r[4] = fmac((C)4, c0[1], c0[2] + c0[0]);        // xx
        r[5] = fmac((C)4, a2[1], a2[2] + a2[0]);        // yy
        r[6] = t;                                       // zz
        r[7] = fmac((C)4, b1[1], b1[2] + b1[0]);        // xy
        r[8] = b0[2] - b0[0];                           // xz
        r[9] = a1[2] - a1[0];                           // yz
    } else {
        r[0] = a0[0];
        r[1] = b0[0];
        r[2] = a1[0];
        r[3] = 0;
        r[4] = c0[0];
        r[5] = a2[0];
        r[6] = 0;
        r[7] = b1[0];
        r[8] = 0;
        r[9] = 0;
    }
    constexpr double sc = L::D == 3 ? 1.0 / 216.0 : 1.0 / 36.0;
    M0 = r[0] * (C)sc;
    static_for<0, 3>([&](auto K) { M1[K] = r[1 + K] * (C)sc; });
    static_for<0, 6>([&](auto K) { M2[K] = r[4 + K] * (C)sc; });
}

// With c_i = g_i + om (feq_i - g_i), feq_i = w_i (3p + 3 e_i.u + 4.5 (e_i.u)^2 - 1.5 u.u):
//   dJ/ds  += sum_i lam_i (g_opp(i) - c_i) + 2 alpha u_x
//   mu_j    = (1-om)(1-s) lam_j + om (Lp + e_j.Lu) + s lam_opp(j) + 2 alpha s e_jx
// where Lp = (1-s) A0 and Lu = (1-s) (3 A + 9 B u - 3 A0 u) are the transposes of the
// moments, written with the moments of w_i lam_i: A0 = sum w lam, A = sum w lam e,
// B = sum w lam e e^T (the per-direction sum Lu = sum (1-s) w lam (3 e + 9 (e.u) e - 3 u)
// regrouped).  Opposite directions share |e.u| and (e.u)^2.
// om = 1/tau rounded once (on the host), sf = s, m = mu, ds = this step's term of dJ/ds
template <int Q, class S, bool SFRAC>
__device__ __forceinline__ void adj_transpose(const typename S::C *lam, const typename S::C *gv, typename S::C sf,
                                              typename S::C om, double alpha, typename S::C *m, double &ds) {
    using L = Lat<Q>;
    using C = typename S::C;
    C p, u[3];
    moments01<L, C>(gv, p, u);
    p = p * (C)(1.0 / 3.0);
    const C al = (C)alpha;
    if constexpr (SFRAC) {
        const C usq = fmac(u[0], u[0], fmac(u[1], u[1], u[2] * u[2]));
        const C X = fmac((C)3, p, (C)-1.5 * usq);
        C acc0 = 0, acc1 = 0;
        static_for<0, Q>([&](auto I) {
            constexpr int i = I, o = L::opp(i);
            if constexpr (i == o) {
                const C c = fmac(om, (C)L::w(i) * X - gv[i], gv[i]);
                acc0 = fmac(lam[i], gv[i] - c, acc0);
            } else if constexpr (i < o) {
                const C eu = edot<L, i>(u);
                const C wt = (C)L::w(i) * fmac((C)4.5 * eu, eu, X);
                const C w3 = (C)(3.0 * L::w(i)) * eu;
                const C ci = fmac(om, (wt + w3) - gv[i], gv[i]);
                const C co = fmac(om, (wt - w3) - gv[o], gv[o]);
                acc0 = fmac(lam[i], gv[o] - ci, acc0);
                acc1 = fmac(lam[o], gv[i] - co, acc1);
            }
        });
        ds = 2.0 * alpha * (double)u[0] + ((double)acc0 + (double)acc1);
    }
    // moments of w lam (B: xx, yy, zz, xy, xz, yz)
    C A0, A[3], B[6];
    wmoments<L, C>(lam, A0, A, B);
    const C ks = (C)1 - sf;
    // V = om Lu (+ 2 alpha s along x), P = om Lp
    const C t3 = (C)3 * A0;
    const C Bu0 = fmac(B[0], u[0], fmac(B[3], u[1], B[4] * u[2]));
    const C Bu1 = fmac(B[3], u[0], fmac(B[1], u[1], B[5] * u[2]));
    const C Bu2 = fmac(B[4], u[0], fmac(B[5], u[1], B[2] * u[2]));
    const C kom = ks * om;
    C V[3];
    V[0] = kom * fmac((C)9, Bu0, fmac((C)3, A[0], -t3 * u[0]));
    V[1] = kom * fmac((C)9, Bu1, fmac((C)3, A[1], -t3 * u[1]));
    V[2] = kom * fmac((C)9, Bu2, fmac((C)3, A[2], -t3 * u[2]));
    if constexpr (SFRAC) V[0] = fmac((C)2 * al, sf, V[0]);
    const C P = kom * A0;
    const C c1 = ((C)1 - om) * ks;
    static_for<0, Q>([&](auto J) {
        constexpr int j = J;
        // E = P + e_z V_z + e_y V_y + e_x V_x, in this order so that directions sharing
        // (e_z) or (e_z, e_y) share the partial sums
        C E = P;
        if constexpr (L::ez(j) > 0) E = E + V[2];
        if constexpr (L::ez(j) < 0) E = E - V[2];
        if constexpr (L::ey(j) > 0) E = E + V[1];
        if constexpr (L::ey(j) < 0) E = E - V[1];
        if constexpr (L::ex(j) > 0) E = E + V[0];
        if constexpr (L::ex(j) < 0) E = E - V[0];
        if constexpr (SFRAC) m[j] = fmac(c1, lam[j], fmac(sf, lam[L::opp(j)], E));
        else m[j] = fmac(c1, lam[j], E);
    });
}

}  // namespace lbm
