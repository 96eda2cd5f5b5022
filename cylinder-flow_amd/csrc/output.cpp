// output.cpp -- device results into the caller's arrays: fields, populations, force records.
//
// The results are gathered in a device buffer of the context and leave it through pinned memory of the
// context, both kept for the next call.  A small result (the monitoring loop's case, where each
// copy and each wait costs ten microseconds) is one copy and one wait.  A large one is cut into
// slices that a few threads take in turn: while one slice crosses the bus into its pinned slot, others are
// copied on to the caller's pages, which a single copy out of device memory does one after the other.
#include <atomic>
#include <cstring>
#include <system_error>

#include "internal.hpp"

using namespace lbm;

namespace {
constexpr size_t SLICE = (size_t)4 << 20;   // bytes of a pinned slot
constexpr int SLOTS = 8;                    // slots, and threads at most
}  // namespace

void output_free(lbm_ctx *c) {
    if (c->out_dev) (void)hipFree(c->out_dev);
    if (c->out_pin) (void)hipHostFree(c->out_pin);
    c->out_dev = nullptr;
    c->out_pin = nullptr;
    c->out_elems = 0;
    c->out_pinned = 0;
    c->hist_copy.clear();
}

// a device buffer of at least `elems` doubles and pinned memory for copies of `bytes` bytes (null where
// there is none to be had: the copies then go straight to the caller's memory)
static hipError_t reserve(lbm_ctx *c, size_t elems, size_t bytes) {
    if (elems > c->out_elems) {
        if (c->out_dev) (void)hipFree(c->out_dev);
        c->out_dev = nullptr;
        c->out_elems = 0;
        const hipError_t e = hipMalloc(&c->out_dev, sizeof(double) * elems);
        if (e != hipSuccess) return e;
        c->out_elems = elems;
    }
    const size_t pinned = bytes <= SLICE ? SLICE : SLICE * SLOTS;
    if (pinned > c->out_pinned) {
        if (c->out_pin) (void)hipHostFree(c->out_pin);
        c->out_pin = nullptr;
        c->out_pinned = 0;
        const hipError_t e = hipHostMalloc((void **)&c->out_pin, pinned, hipHostMallocDefault);
        if (e != hipSuccess) {
            c->out_pin = nullptr;
            (void)hipGetLastError();
            return hipSuccess;
        }
        c->out_pinned = pinned;
    }
    return hipSuccess;
}

// `bytes` of device memory into dst, after the stream's work so far; returns when they are there
static hipError_t copy_out(lbm_ctx *c, void *dst, const void *src, size_t bytes) {
    if (!c->out_pin) {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream);
        return e == hipSuccess ? hipStreamSynchronize(c->stream) : e;
    }
    if (bytes <= SLICE) {
        hipError_t e = hipMemcpyAsync(c->out_pin, src, bytes, hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        if (e == hipSuccess) std::memcpy(dst, c->out_pin, bytes);
        return e;
    }
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const size_t slices = (bytes + SLICE - 1) / SLICE;
    std::atomic<int> failed{(int)hipSuccess};
    auto work = [&](int t, bool own) {   // slices t, t + SLOTS, ... through slot t
        hipError_t r = own ? hipSetDevice(dev) : hipSuccess;
        hipEvent_t ev = nullptr;
        if (r == hipSuccess) r = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        char *const slot = (char *)c->out_pin + SLICE * (size_t)t;
        for (size_t s = (size_t)t; s < slices && r == hipSuccess && failed.load() == (int)hipSuccess; s += SLOTS) {
            const size_t off = s * SLICE, n = std::min(SLICE, bytes - off);
            r = hipMemcpyAsync(slot, (const char *)src + off, n, hipMemcpyDeviceToHost, c->stream);
            if (r == hipSuccess) r = hipEventRecord(ev, c->stream);
            if (r == hipSuccess) r = hipEventSynchronize(ev);
            if (r == hipSuccess) std::memcpy((char *)dst + off, slot, n);
        }
        if (ev) (void)hipEventDestroy(ev);
        if (r != hipSuccess) failed.store((int)r);
    };
    std::thread th[SLOTS];
    const int want = (int)std::min<size_t>(SLOTS, slices);
    int started = 1;   // thread 0 is this one
    try {
        for (; started < want; started++) th[started] = std::thread(work, started, true);
    } catch (const std::system_error &) {   // no more threads: their slices are done below
    }
    work(0, false);
    for (int t = 1; t < started; t++) th[t].join();
    for (int t = started; t < want; t++) work(t, false);
    e = (hipError_t)failed.load();
    const hipError_t e2 = hipStreamSynchronize(c->stream);
    return e != hipSuccess ? e : e2;
}

// the requested fields (null: not wanted) of the current state, in c's order p, u, v, w
hipError_t output_fields(lbm_ctx *c, double *const *outs) {
    unsigned want = 0;
    int n = 0;
    for (int k = 0; k < 4; k++)
        if (outs[k]) {
            want |= 1u << k;
            n++;
        }
    if (n == 0) return hipSuccess;
    const bool ref = c->cfg.bc_mode != LBM_BC_PLAIN;
    const size_t bytes = sizeof(double) * c->N;
    auto gather = [&](unsigned mask) {
        return ref ? ref_fields(c->rg, c->rmac, c->out_dev, mask, c->stream)
                   : plain_fields(c->macros, c->flags, c->out_dev, mask, c->geo, c->stream);
    };
    if (bytes * n <= SLICE) {   // all of them in one kernel, one copy and one wait
        hipError_t e = reserve(c, c->N * n, bytes * n);
        if (e == hipSuccess) e = gather(want);
        if (e == hipSuccess && !c->out_pin) {
            const double *from = c->out_dev;
            for (int k = 0; k < 4 && e == hipSuccess; k++)
                if (outs[k]) {
                    e = copy_out(c, outs[k], from, bytes);
                    from += c->N;
                }
            return e;
        }
        if (e == hipSuccess) e = hipMemcpyAsync(c->out_pin, c->out_dev, bytes * n, hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        if (e != hipSuccess) return e;
        const double *p = c->out_pin;
        for (int k = 0; k < 4; k++)
            if (outs[k]) {
                std::memcpy(outs[k], p, bytes);
                p += c->N;
            }
        return hipSuccess;
    }
    hipError_t e = reserve(c, c->N, bytes);
    for (int k = 0; k < 4 && e == hipSuccess; k++) {
        if (!outs[k]) continue;
        e = gather(1u << k);
        if (e == hipSuccess) e = copy_out(c, outs[k], c->out_dev, bytes);
    }
    return e;
}

// a device buffer of N doubles for one direction's populations, and its copy to dst
hipError_t output_stage(lbm_ctx *c, double **dev) {
    const hipError_t e = reserve(c, c->N, sizeof(double) * c->N);
    *dev = c->out_dev;
    return e;
}
hipError_t output_staged(lbm_ctx *c, double *dst) { return copy_out(c, dst, c->out_dev, sizeof(double) * c->N); }

// The force records so far, on the host: the context keeps a copy, and only the records since the last
// call cross the bus (a program that reads its record at every output would move all of it each time).
hipError_t output_forces(lbm_ctx *c) {
    const size_t have = c->hist_copy.size() / 4, all = (size_t)c->nrec;
    if (have >= all) return hipStreamSynchronize(c->stream);   // callers may count on the stream being drained
    const size_t bytes = sizeof(double) * 4 * (all - have);
    hipError_t e = reserve(c, 0, bytes);
    if (e != hipSuccess) return e;
    try {
        c->hist_copy.resize(4 * all);
    } catch (const std::bad_alloc &) {
        return hipErrorOutOfMemory;
    }
    e = copy_out(c, c->hist_copy.data() + 4 * have, c->hist + 4 * have, bytes);
    if (e != hipSuccess) c->hist_copy.resize(4 * have);
    return e;
}
