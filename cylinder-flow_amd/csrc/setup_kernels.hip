// setup_kernels.hip -- initialisation of the plain mode's node arrays on the device: node flags from the
// body formula or the mask, the padded solid fraction, and the per-row and per-block predicates that the
// host's lists are built from.  (3D MPI+KOKKOS+MPIIO/lbm.cpp:238 for the "usr" formula.)  On the host the
// same classification, up to 26 neighbour tests per node, took 78 of the 80 ms of an initialisation at
// 192x96x96 (now 1.9 ms in all) and 0.5 of 0.77 ms at 400x100 (0.20).  One lane per node in blocks of 256
// along a row: bound by the flags' bytes and by launches, so nothing is staged.
#include "internal.hpp"
#include "lattice.hpp"

namespace lbm {

// solid or fluid; the padding of a row is solid.  Clears the counts of the next launch.
__global__ void __launch_bounds__(256) k_setup_solid(uint8_t *__restrict__ flags, const uint8_t *__restrict__ mask, SetupBody b, Geo g,
                                                     int D, unsigned *__restrict__ counts) {
    if (blockIdx.x + blockIdx.y + blockIdx.z == 0 && threadIdx.x < 3) counts[threadIdx.x] = 0u;
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, z = blockIdx.z;
    if (x >= g.nxp) return;
    const size_t row = (size_t)y + (size_t)g.ny * z;
    bool solid = x >= g.nx;
    if (!solid && mask) solid = mask[(size_t)x + (size_t)g.nx * row] != 0;
    if (!solid && !mask && (b.kind == LBM_BODY_SPHERE || b.kind == LBM_BODY_ZCYL)) {
        const double dx = (double)x - b.cx, dy = (double)y - b.cy;
        double r = dx * dx + dy * dy;
        if (D == 3 && b.kind == LBM_BODY_SPHERE) {
            const double dz = (double)z - b.cz;
            r = r + dz * dz;
        }
        solid = r <= b.r2;
    }
    flags[(size_t)x + (size_t)g.nxp * row] = solid ? FL_SOLID : FL_FLUID;
}

__device__ __forceinline__ void wave_count(bool v, unsigned *dst) {
    const unsigned long long m = __builtin_amdgcn_ballot_w64(v);
    if ((threadIdx.x & 63) == 0 && m) atomicAdd(dst, (unsigned)__builtin_popcountll(m));
}

// fluid nodes with a solid neighbour become FL_NEAR (in place: neighbours are only tested for FL_SOLID, which
// no lane writes); counts: the solid and the near nodes and those of the fix list
template <int Q>
__global__ void __launch_bounds__(256) k_setup_near(uint8_t *flags, const double *__restrict__ sfrac, Geo g, SetupFix fix,
                                                    unsigned *__restrict__ counts) {
    using L = Lat<Q>;
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, z = blockIdx.z;
    const bool in = x < g.nx;
    const size_t row = (size_t)y + (size_t)g.ny * z, node = (size_t)(in ? x : 0) + (size_t)g.nxp * row;
    const bool solid = in && flags[node] == FL_SOLID, fluid = in && !solid;
    bool near = false, to_fix = false;
    if (fluid) {
        static_for<1, Q>([&](auto I) {
            constexpr int i = I;
            int sx = x - L::ex(i), sy = y - L::ey(i), sz = z - L::ez(i);
            if (g.xper) sx = sx < 0 ? sx + g.nx : (sx >= g.nx ? sx - g.nx : sx);
            if (g.yper) sy = sy < 0 ? sy + g.ny : (sy >= g.ny ? sy - g.ny : sy);
            if (g.zper) sz = sz < 0 ? sz + g.nz : (sz >= g.nz ? sz - g.nz : sz);
            if ((unsigned)sx < (unsigned)g.nx && (unsigned)sy < (unsigned)g.ny && (unsigned)sz < (unsigned)g.nz)
                near = near || flags[(size_t)sx + (size_t)g.nxp * ((size_t)sy + (size_t)g.ny * sz)] == FL_SOLID;
        });
        if (near) flags[node] = FL_NEAR;
        const bool sfr = sfrac && sfrac[(size_t)x + (size_t)g.nx * row] > 0.0;
        to_fix = fix.all || sfr || fix_edge(g, fix.V, x) || (near && (fix_end_lane(g, fix.V, x) || !fix.same_offsets));
    }
    wave_count(solid, counts);
    wave_count(near, counts + 1);
    wave_count(fluid && to_fix, counts + 2);
}

// per block of bx nodes of a row (gx per row): 1 when one of them carries force (next to the mask, or
// fluid with a solid fraction)
__global__ void __launch_bounds__(256) k_setup_forced(const uint8_t *__restrict__ flags, const double *__restrict__ sfrac,
                                                      uint8_t *__restrict__ out, Geo g) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const size_t row = (size_t)blockIdx.y + (size_t)g.ny * blockIdx.z;
    bool f = false;
    if (x < g.nx) {
        const uint8_t fl = flags[(size_t)x + (size_t)g.nxp * row];
        f = fl == FL_NEAR || (sfrac && fl != FL_SOLID && sfrac[(size_t)x + (size_t)g.nx * row] > 0.0);
    }
    const int any = __syncthreads_or(f);
    if (threadIdx.x == 0) out[blockIdx.x + (size_t)gridDim.x * row] = any ? 1 : 0;
}

// per row: 1 when every node is fluid with no solid neighbour
__global__ void __launch_bounds__(256) k_setup_clean(const uint8_t *__restrict__ flags, uint8_t *__restrict__ clean,
                                                     uint8_t *__restrict__ copy, Geo g) {
    const size_t row = (size_t)blockIdx.x + (size_t)g.ny * blockIdx.y;
    bool bad = false;
    for (int x = threadIdx.x; x < g.nx; x += 256) bad = bad || flags[(size_t)x + (size_t)g.nxp * row] != FL_FLUID;
    const int any = __syncthreads_or(bad);
    if (threadIdx.x == 0) clean[row] = copy[row] = any ? 0 : 1;
}

__global__ void __launch_bounds__(256) k_setup_links9(const uint8_t *__restrict__ flags, uint16_t *__restrict__ lk, Geo g) {
    using L = Lat<9>;
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
    if (x >= g.nxp) return;
    const size_t node = (size_t)x + (size_t)g.nxp * y;
    const bool wallrow = !g.yper && (y == 0 || y == g.ny - 1);
    const uint8_t fl = flags[node];   // padding nodes are solid
    uint32_t b = 0;
    if (fl != FL_SOLID && (wallrow || fl == FL_NEAR))
        static_for<1, 9>([&](auto I) {
            constexpr int i = I;
            constexpr int ex = L::ex(i), ey = L::ey(i);
            if (ex > 0 && x == 0 && !g.xper) return;   // Zou-He unknown
            int sx = x - ex, sy = y - ey;
            if (g.yper) sy = sy < 0 ? sy + g.ny : (sy >= g.ny ? sy - g.ny : sy);
            if ((unsigned)sy >= (unsigned)g.ny) {      // wall
                b |= 1u << (7 + i);
                return;
            }
            if (g.xper) sx = sx < 0 ? sx + g.nx : (sx >= g.nx ? sx - g.nx : sx);
            else if (sx == g.nx) sx = x;               // outlet clamp
            if (flags[(size_t)sx + (size_t)g.nxp * sy] == FL_SOLID) b |= 1u << (i - 1);
        });
    lk[node] = (uint16_t)b;
}

template <class C>
__global__ void __launch_bounds__(256) k_setup_sfrac(const double *__restrict__ in, C *__restrict__ out, Geo g) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, z = blockIdx.z;
    if (x >= g.nxp) return;
    const size_t row = (size_t)y + (size_t)g.ny * z;
    out[(size_t)x + (size_t)g.nxp * row] = x < g.nx ? (C)in[(size_t)x + (size_t)g.nx * row] : (C)0;
}

static dim3 row_blocks(const Geo &g) { return dim3((unsigned)((g.nxp + 255) / 256), (unsigned)g.ny, (unsigned)g.nz); }

hipError_t setup_flags(int Q, uint8_t *flags, const uint8_t *mask, const double *sfrac, const SetupBody &b, const SetupFix &fix,
                       const Geo &g, unsigned *counts, hipStream_t s) {
    hipLaunchKernelGGL(k_setup_solid, row_blocks(g), dim3(256), 0, s, flags, mask, b, g, Q == 9 ? 2 : 3, counts);
    if (Q == 9) hipLaunchKernelGGL(k_setup_near<9>, row_blocks(g), dim3(256), 0, s, flags, sfrac, g, fix, counts);
    else hipLaunchKernelGGL(k_setup_near<27>, row_blocks(g), dim3(256), 0, s, flags, sfrac, g, fix, counts);
    return hipGetLastError();
}

hipError_t setup_forced(const uint8_t *flags, const double *sfrac, uint8_t *out, Shape blk, const Geo &g, hipStream_t s) {
    hipLaunchKernelGGL(k_setup_forced, dim3((unsigned)blk.gx, (unsigned)g.ny, (unsigned)g.nz), dim3((unsigned)blk.bx), 0, s, flags, sfrac,
                       out, g);
    return hipGetLastError();
}

hipError_t setup_clean(const uint8_t *flags, uint8_t *clean, uint8_t *copy, const Geo &g, hipStream_t s) {
    hipLaunchKernelGGL(k_setup_clean, dim3((unsigned)g.ny, (unsigned)g.nz), dim3(256), 0, s, flags, clean, copy, g);
    return hipGetLastError();
}

hipError_t setup_sfrac(int prec, const double *in, void *out, const Geo &g, hipStream_t s) {
    if (prec == LBM_FP64) hipLaunchKernelGGL(k_setup_sfrac<double>, row_blocks(g), dim3(256), 0, s, in, (double *)out, g);
    else hipLaunchKernelGGL(k_setup_sfrac<float>, row_blocks(g), dim3(256), 0, s, in, (float *)out, g);
    return hipGetLastError();
}

hipError_t setup_links9(const uint8_t *flags, uint16_t *lk, const Geo &g, hipStream_t s) {
    hipLaunchKernelGGL(k_setup_links9, row_blocks(g), dim3(256), 0, s, flags, lk, g);
    return hipGetLastError();
}

}  // namespace lbm
