// Side streams on which the buckets of one path-list call run next to each other (no counterpart in the reference, whose
// stage runs one chunk after the other). A bucket of a few hundred paths fills a fraction of the chip, and each of its
// kernels lasts as long as one workgroup: run side by side the buckets of a small list cost little more than the longest.
// Steps, us: small Cu cluster (2, 3 and 4 legs) 324 -> 190, MD batch of 64 frames 3400 -> 3200, FP64 refinement 1550 ->
// 1350, two-edge alloy (10 buckets) 12.1 -> 11.4 ms.
#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>

#include "fm_internal.h"

namespace fm {

namespace {
constexpr int MAX_DEV = 64, POOL_MAX = 16;     // released sets kept per device for the next plan
std::mutex g_mutex;
std::vector<fm_overlap *> g_free[MAX_DEV];

void destroy(fm_overlap *o) {
    for (hipStream_t s : o->side)
        if (s) (void)hipStreamDestroy(s);
    for (hipEvent_t e : o->join)
        if (e) (void)hipEventDestroy(e);
    if (o->fork) (void)hipEventDestroy(o->fork);
    delete o;
}
}  // namespace

Lanes::Lanes(fm_overlap *o_, hipStream_t st_, int want) : o(o_), st(st_) {
    int dev = -1;
    if (!o || want < 2 || hipGetDevice(&dev) != hipSuccess || dev != o->dev) return;
    const int side = want - 1 < FM_SIDE ? want - 1 : FM_SIDE;
    for (int i = 0; i < side; ++i) {
        // a side stream that another stream's capture has drawn in would put this call's work into that graph
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone, mine = hipStreamCaptureStatusNone;
        unsigned long long id = 0, my_id = 0;
        if (hipStreamGetCaptureInfo(o->side[i], &cs, &id) != hipSuccess) return;
        if (cs == hipStreamCaptureStatusNone) continue;
        if (!st || hipStreamGetCaptureInfo(st, &mine, &my_id) != hipSuccess || mine != cs || my_id != id) return;
    }
    if ((err = hipEventRecord(o->fork, st)) != hipSuccess) return;
    for (int i = 0; i < side; ++i) {
        if ((err = hipStreamWaitEvent(o->side[i], o->fork, 0)) != hipSuccess) return;
        n = 2 + i;
    }
}

hipError_t Lanes::join() {
    for (int i = 0; i + 1 < n; ++i) {
        hipError_t e = hipEventRecord(o->join[i], o->side[i]);
        if (e == hipSuccess) e = hipStreamWaitEvent(st, o->join[i], 0);
        if (e != hipSuccess && err == hipSuccess) err = e;
    }
    n = 1;
    return err;
}

std::vector<int> lanes_of(int nbucket, const int32_t *offset, const int32_t *nleg, int nlane) {
    std::vector<int> lane(nbucket > 0 ? nbucket : 0, 0), order;
    double load[1 + FM_SIDE] = {};
    auto cost = [&](int b) { return (double)(offset[b + 1] - offset[b]) * nleg[b]; };
    for (int b = 0; b < nbucket; ++b) {
        size_t at = 0;
        while (at < order.size() && cost(order[at]) >= cost(b)) ++at;
        order.insert(order.begin() + at, b);
    }
    for (int b : order) {
        int l = 0;
        for (int i = 1; i < nlane; ++i)
            if (load[i] < load[l]) l = i;
        lane[b] = l;
        load[l] += cost(b);
    }
    return lane;
}

}  // namespace fm

extern "C" {

fm_overlap *fm_overlap_acquire(void) {
    using namespace fm;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEV) return nullptr;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (!g_free[dev].empty()) {
            fm_overlap *o = g_free[dev].back();
            g_free[dev].pop_back();
            return o;
        }
    }
    fm_overlap *o = new (std::nothrow) fm_overlap();
    if (!o) return nullptr;
    o->dev = dev;
    bool ok = hipEventCreateWithFlags(&o->fork, hipEventDisableTiming) == hipSuccess;
    for (int i = 0; i < FM_SIDE; ++i)
        ok = ok && hipStreamCreateWithFlags(&o->side[i], hipStreamNonBlocking) == hipSuccess &&
             hipEventCreateWithFlags(&o->join[i], hipEventDisableTiming) == hipSuccess;
    if (ok) return o;
    destroy(o);
    return nullptr;
}

void fm_overlap_release(fm_overlap *o) {
    using namespace fm;
    if (!o) return;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (g_free[o->dev].size() < POOL_MAX) {
            try {
                g_free[o->dev].push_back(o);
                return;
            } catch (...) {
            }
        }
    }
    destroy(o);
}

}  // extern "C"
