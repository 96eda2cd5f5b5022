// pair.cpp -- host side of the two-step kernel (pair_kernel.hpp): where it applies, the bounce words
// and the column runs.
#include <algorithm>
#include <cstdlib>

#include "internal.hpp"
#include "lattice.hpp"

namespace lbm {

PairOps pair_ops_f64();
PairOps pair_ops_f32();
PairOps pair_ops_f16();
PairOps pair_ops_bf16();

PairOps pair_ops(int prec) {
    return prec == LBM_FP64 ? pair_ops_f64() : prec == LBM_FP32 ? pair_ops_f32() : prec == LBM_FP16S ? pair_ops_f16() : pair_ops_bf16();
}

void pair_free(PairPlan &p) {
    for (void *q : {(void *)p.bw, (void *)p.tflag, (void *)p.link, (void *)p.linklk, (void *)p.link_slot, (void *)p.fblk, (void *)p.partials, (void *)p.seg, (void *)p.trip})
        if (q) (void)hipFree(q);
    p = PairPlan{};
}

template <class T>
static hipError_t upload(T *&dst, const std::vector<T> &src) {
    hipError_t e = hipMalloc(&dst, sizeof(T) * std::max<size_t>(src.size(), 1));
    if (e == hipSuccess && !src.empty()) e = hipMemcpy(dst, src.data(), sizeof(T) * src.size(), hipMemcpyHostToDevice);
    return e;
}

// Whether two steps per pass take less time than two one-step launches: a pass takes 9 us (FP64), 5 (FP32) or
// 4.25 (16 bits) per plane of work and round, a one-step launch a few us and then its share per 1000
// padded nodes; in 16 bits that holds for the packed kernel alone (dense mode and a fix-up list are
// slower at every size measured).  Two columns of few planes each redo most of their first step: us per
// step, one step per launch / two steps per pass, on 40 domains from 24x16x16 to 320x140x140 (the constants
// follow them): FP64 24x16x16 7.2 / 12.1, 40x123x30 18.8 / 21.9, 96x48x48 22.4 / 21.6, 125x67x45 33.5 / 30.5,
// 320x140x140 548 / 377; FP32 61x23x22 7.0 / 7.9, 33x53x28 8.3 / 8.4, 125x67x45 19.2 / 14.1; FP16 packed
// 222x17x124 15.8 / 18.4, 320x140x140 120 / 128 (two rounds), 192x96x96 38.3 / 35.1.
static bool pair_pays(int prec, const Geo &g, long cost, bool packed) {
    const double k = 1e-3 * (double)g.plane;
    if (prec == LBM_FP64) return 9.0 * cost / 2 < 5.5 + 0.068 * k;
    if (prec == LBM_FP32) return 5.0 * cost / 2 < 6.2 + 0.031 * k;
    return !packed || 4.25 * cost / 2 < 4.0 + 0.0195 * k;
}

hipError_t pair_plan(PairPlan &p, int prec, const Geo &g, const uint8_t *flags, bool same_offsets, bool packed,
                     const std::vector<uint32_t> &near_nodes, const std::vector<int> &block_slot, Shape blk, hipStream_t s) {
    pair_free(p);
    // LBM_TWO_STEPS=0 keeps one step per launch, 1 takes two per pass whether or not that pays; any switch
    // that selects among the one-step kernels keeps one.  Opposite directions must share their storage offset (a bounced value is taken as
    // stored), the rows must be interleaved, and the buffers' byte offsets must fit 32 bits: the
    // three planes a pull spans, with periodic z the whole state.
    const char *env = std::getenv("LBM_TWO_STEPS");
    if (env && env[0] == '0') return hipSuccess;
    for (const char *k : {"LBM_FORCE_SLOW_PATH", "LBM_DENSE", "LBM_ALIGNED_PULL", "LBM_NODES_PER_LANE", "LBM_FAST_BLOCKS_PER_CU"})
        if (std::getenv(k)) return hipSuccess;
    const size_t esz = prec == LBM_FP64 ? 8 : prec == LBM_FP32 ? 4 : 2;
    const double planeb = (double)g.rs * g.ny * esz, limit = 4294967296.0;
    if (!same_offsets || g.ds != (size_t)g.nxp || planeb * (g.zper ? g.nz : 3) >= limit) return hipSuccess;
    const PairOps ops = pair_ops(prec);
    int dev = 0, lds = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    if ((size_t)lds < ops.lds || ops.prepare() != hipSuccess) return hipSuccess;
    p.tiles_x = (g.nx + ops.wx - 1) / ops.wx;
    p.tiles_y = (g.ny + ops.wy - 1) / ops.wy;
    // planes per block (one block per CU at a time): c planes take c + 2 first steps and c second ones
    // in c + 3 passes, about c + 2 planes of work; the least (rounds of the CUs) x (c + 2).  Measured on
    // 512x256x256 in FP32, 256 columns: 871 us per step in one run of 256 planes, 879 in two, 885 in 8;
    // on 256x128x128, 64 columns: 116 in four runs (one round), 124 in eight
    const long tiles = (long)p.tiles_x * p.tiles_y;
    long best = -1;
    for (int n = 1; n <= g.nz; n++) {
        const int c = (g.nz + n - 1) / n, m = (g.nz + c - 1) / c;
        const long cost = ((tiles * m + cus - 1) / cus) * (c + 2);
        if (best < 0 || cost < best) {
            best = cost;
            p.cz = c;
            p.chunks = m;
        }
    }
    if (!(env && env[0] == '1') && !pair_pays(prec, g, best, packed)) return hipSuccess;
    // bounce words, column bits and the links of the listed nodes, on the device
    const size_t words = (size_t)((g.nz + 31) / 32) * (size_t)tiles;
    if (near_nodes.size() > (size_t)INT32_MAX) return hipSuccess;
    const bool per_block = !block_slot.empty();
    p.nlink = p.nslots = per_block ? 0 : (int)near_nodes.size();
    std::vector<int> slot((size_t)p.nlink);
    for (size_t k = 0; k < slot.size(); k++) slot[k] = (int)k;
    std::vector<uint32_t> fblk;
    for (size_t b = 0; b < block_slot.size(); b++)
        if (block_slot[b] >= 0) fblk.push_back((uint32_t)b);   // slots count up in block order
    if (!fblk.empty()) {
        p.nslots = (int)fblk.size();
        p.fbx = blk.bx;
        p.fgx = blk.gx;
        e = upload(p.fblk, fblk);
    }
    if (e == hipSuccess) e = hipMalloc(&p.bw, sizeof(uint32_t) * g.plane);
    if (e == hipSuccess) e = hipMalloc(&p.tflag, sizeof(uint32_t) * words);
    if (e == hipSuccess && p.nlink) {
        e = upload(p.link, near_nodes);
        if (e == hipSuccess) e = upload(p.link_slot, slot);
        if (e == hipSuccess) e = hipMalloc(&p.linklk, sizeof(uint32_t) * (size_t)p.nlink);
    }
    // the nodes next to the mask by segments of 64
    std::vector<unsigned long long> masks(g.plane / 64);
    unsigned long long *dmasks = nullptr;
    if (e == hipSuccess) e = hipMalloc(&dmasks, sizeof(masks[0]) * masks.size());
    if (e == hipSuccess) e = pair_words(p, ops, flags, dmasks, g, s);
    if (e == hipSuccess) e = hipMemcpyAsync(masks.data(), dmasks, sizeof(masks[0]) * masks.size(), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (dmasks) (void)hipFree(dmasks);
    if (e == hipSuccess) {
        std::vector<PairSeg> seg(masks.size());
        size_t n = 0;
        for (size_t k = 0; k < seg.size(); k++) {
            seg[k] = {(uint32_t)n, (uint32_t)masks[k], (uint32_t)(masks[k] >> 32), 0u};
            n += (size_t)__builtin_popcountll(masks[k]);
        }
        // The force of a second step is summed in the pass, except in 16 bits next to the packed one-step
        // kernel, where its instructions cost more than they save: 512x256x256, the force every step, one
        // launch per step / two steps per pass with it, FP64 2671 / 1753 us per step, FP32 1242 / 864, FP16
        // 649 / 743.  (The sums are addressed in bytes of 32 bits.)
        if (n * 24 < ((size_t)1 << 32) && (prec == LBM_FP64 || prec == LBM_FP32 || !packed)) {
            p.nnear = (int)n;
            e = upload(p.seg, seg);
            if (e == hipSuccess && per_block) e = hipMalloc(&p.trip, 24 * std::max<size_t>(n, 1));
        }
    }
    if (e == hipSuccess) e = hipMalloc(&p.partials, force_bytes(p.nslots));
    if (e != hipSuccess) {
        pair_free(p);
        if (e != hipErrorOutOfMemory) return e;
        (void)hipGetLastError();   // no room for the words: one step per launch
        return hipSuccess;
    }
    p.on = true;
    return hipSuccess;
}

}  // namespace lbm
