// pair_words.hip -- the two-step kernel's bounce words, from the node flags (pair_kernel.hpp).
#include "internal.hpp"
#include "lattice.hpp"

namespace lbm {

// the directions a fluid node pulls across a wall or from a solid node, with the pull's classification:
// inlet unknowns first, then walls, then the outlet's clamped or the periodic source
__device__ __forceinline__ void bounce_word(const uint8_t *__restrict__ flags, const Geo &g, int x, int y, int z, uint8_t fl,
                                            uint32_t &wall, uint32_t &mask) {
    using L = Lat<27>;
    wall = mask = 0u;
    static_for<1, 27>([&](auto I) {
        constexpr int i = I;
        constexpr int ex = L::ex(i), ey = L::ey(i), ez = L::ez(i);
        int sx = x - ex, sy = y - ey, sz = z - ez;
        if (ex > 0 && x == 0 && !g.xper) return;
        if (g.yper) sy = sy < 0 ? sy + g.ny : (sy >= g.ny ? sy - g.ny : sy);
        if (g.zper) sz = sz < 0 ? sz + g.nz : (sz >= g.nz ? sz - g.nz : sz);
        if ((unsigned)sy >= (unsigned)g.ny || (unsigned)sz >= (unsigned)g.nz) {
            wall |= 1u << i;
            return;
        }
        if (g.xper) sx = sx < 0 ? sx + g.nx : (sx >= g.nx ? sx - g.nx : sx);
        else if (sx == g.nx) sx = g.nx - 1;
        if (fl == FL_NEAR && flags[(size_t)sx + (size_t)g.nxp * ((size_t)sy + (size_t)g.ny * sz)] == FL_SOLID) mask |= 1u << i;
    });
}

// bw of every node; a bit per column and plane whose positions [X0 - 1, X0 + wx] x [Y0 - 1, Y0 + wy]
// (also through a periodic axis) hold a non-zero word
__global__ void __launch_bounds__(256) k_pair_words(const uint8_t *__restrict__ flags, uint32_t *__restrict__ bw,
                                                    uint32_t *__restrict__ tflag, unsigned long long *__restrict__ masks, Geo g,
                                                    int wx, int wy, int tiles_x, int tiles_y) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, z = blockIdx.z;
    if (x >= g.nxp) return;
    const size_t node = (size_t)x + (size_t)g.nxp * ((size_t)y + (size_t)g.ny * z);
    uint32_t wall = 0, mask = 0;
    const uint8_t fl = flags[node];   // padding nodes are solid
    const unsigned long long near = __builtin_amdgcn_ballot_w64(fl == FL_NEAR);   // (rows are multiples of 64 nodes)
    if ((threadIdx.x & 63u) == 0) masks[node >> 6] = near;
    const bool wallrow = (!g.yper && (y == 0 || y == g.ny - 1)) || (!g.zper && (z == 0 || z == g.nz - 1));
    if (fl != FL_SOLID && (wallrow || fl == FL_NEAR)) bounce_word(flags, g, x, y, z, fl, wall, mask);
    bw[node] = wall | mask;
    if ((wall | mask) == 0u && fl != FL_NEAR) return;   // (a node next to the mask has a force slot, links or not)
    const int words = (g.nz + 31) / 32, tx = x / wx, ty = y / wy;
    for (int j = -1; j <= 1; j++)
        for (int i = -1; i <= 1; i++) {
            int cx = tx + i, cy = ty + j;
            if (cx < 0 && g.xper) cx = tiles_x - 1;
            if (cx >= tiles_x && g.xper) cx = 0;
            if (cy < 0 && g.yper) cy = tiles_y - 1;
            if (cy >= tiles_y && g.yper) cy = 0;
            if (cx < 0 || cx >= tiles_x || cy < 0 || cy >= tiles_y) continue;
            // in the column's rim: next to it, or across a periodic edge (the last column may be short)
            const bool nx_ = i == 0 || (i < 0 ? x % wx == 0 : x % wx == wx - 1 || x == g.nx - 1);
            const bool ny_ = j == 0 || (j < 0 ? y % wy == 0 : y % wy == wy - 1 || y == g.ny - 1);
            uint32_t *const w = &tflag[((size_t)cy * tiles_x + cx) * words + z / 32];
            const uint32_t bit = 1u << (z % 32);
            if (nx_ && ny_ && (*(volatile uint32_t *)w & bit) == 0u) atomicOr(w, bit);
        }
}

__global__ void __launch_bounds__(256) k_pair_links(const uint8_t *__restrict__ flags, const uint32_t *__restrict__ list, int n,
                                                    uint32_t *__restrict__ lk, Geo g) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const uint32_t node = list[j], row = node / (uint32_t)g.nxp;
    uint32_t wall, mask;
    bounce_word(flags, g, (int)(node - row * (uint32_t)g.nxp), (int)(row % (uint32_t)g.ny), (int)(row / (uint32_t)g.ny), FL_NEAR,
                wall, mask);
    lk[j] = mask;
}

hipError_t pair_words(const PairPlan &p, const PairOps &ops, const uint8_t *flags, unsigned long long *masks, const Geo &g,
                      hipStream_t s) {
    hipError_t e = hipMemsetAsync(p.tflag, 0, sizeof(uint32_t) * (size_t)((g.nz + 31) / 32) * p.tiles_x * p.tiles_y, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_pair_words, dim3((unsigned)((g.nxp + 255) / 256), (unsigned)g.ny, (unsigned)g.nz), dim3(256), 0, s, flags,
                       p.bw, p.tflag, masks, g, ops.wx, ops.wy, p.tiles_x, p.tiles_y);
    if ((e = hipGetLastError()) != hipSuccess || p.nlink == 0) return e;
    hipLaunchKernelGGL(k_pair_links, dim3((unsigned)((p.nlink + 255) / 256)), dim3(256), 0, s, flags, p.link, p.nlink, p.linklk, g);
    return hipGetLastError();
}

}  // namespace lbm
