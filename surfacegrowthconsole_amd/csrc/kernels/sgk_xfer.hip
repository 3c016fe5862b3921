// sgk_xfer.hip - state transfer through pinned slots that the kernels read and write (sgk_xfer.h).
#include "sgk_xfer.h"

#include <algorithm>
#include <cstring>
#include <thread>
#include <vector>

namespace sgk {

namespace {

constexpr int kMaxArrays = 3;

// The arrays of one transfer, their host values laid end to end; array k starts at value begin[k].
struct Layout {
    const void *dev[kMaxArrays];
    unsigned long long begin[kMaxArrays + 1];
    XferLayout layout[kMaxArrays];
    bool wide[kMaxArrays];
};

// Where value j of an array lies on the device.
__device__ __forceinline__ unsigned long long place(XferLayout l, unsigned long long j, unsigned long long count) {
    if (l == XferLayout::plain) return j;
    if (l == XferLayout::energy) return 4 * j + 3;
    const unsigned int atom = (unsigned int)(j / 3), d = (unsigned int)(j - 3ull * atom);
    return d * (count / 3) + atom;
}

// Values [at, at + m) between the arrays and a slot, one per thread: the slot's side of a wave is one
// run of 512 (256) bytes, which is what the link to the host asks for, and the gather by atom stays in
// the device's caches.
template <class H, bool OUT>
__global__ __launch_bounds__(256) void k_xfer(Layout a, unsigned long long at, unsigned int m, H *__restrict__ slot) {
    const unsigned int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    const unsigned long long j = at + i;
    const int k = j < a.begin[1] ? 0 : j < a.begin[2] ? 1 : 2;
    const unsigned long long q = place(a.layout[k], j - a.begin[k], a.begin[k + 1] - a.begin[k]);
    if constexpr (OUT) {
        slot[i] = a.wide[k] ? (H)((const double *)a.dev[k])[q] : (H)((const float *)a.dev[k])[q];
    } else {
        if (a.wide[k])
            ((double *)a.dev[k])[q] = (double)slot[i];
        else
            ((float *)a.dev[k])[q] = (float)slot[i];
    }
}

// The owner's device while a transfer runs: the caller's thread may have another one set.
struct OnDevice {
    int before = -1, device;
    explicit OnDevice(int d) : device(d) {
        if (hipGetDevice(&before) == hipSuccess && before != device) (void)hipSetDevice(device);
    }
    ~OnDevice() {
        if (before >= 0 && before != device) (void)hipSetDevice(before);
    }
};

template <class H, bool OUT>
struct Transfer {
    hipStream_t s;
    const XferArray *arrays;
    int n;
    Layout lay;
    size_t slot;  // values of a slot

    // A slot's values and the host arrays they belong to.
    void host_copy(size_t at, size_t m, H *p) const {
        for (int k = 0; k < n; ++k) {
            const size_t b = (size_t)lay.begin[k], lo = std::max(at, b), hi = std::min(at + m, (size_t)lay.begin[k + 1]);
            if (lo >= hi) continue;
            H *h = (H *)arrays[k].host + (lo - b), *q = p + (lo - at);
            std::memcpy(OUT ? h : q, OUT ? q : h, (hi - lo) * sizeof(H));
        }
    }
    hipError_t issue(size_t at, size_t m, H *p, hipEvent_t ev) const {
        hipLaunchKernelGGL((k_xfer<H, OUT>), dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, lay,
                           (unsigned long long)at, (unsigned int)m, p);
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? hipEventRecord(ev, s) : e;
    }
    // Values [lo, hi) through two slots.  No kernel still uses a slot on return, also after an error.
    hipError_t part(size_t lo, size_t hi, H *slots, hipEvent_t *ev) const {
        const size_t pieces = (hi - lo + slot - 1) / slot;
        auto at = [&](size_t k) { return lo + k * slot; };
        auto len = [&](size_t k) { return std::min(slot, hi - at(k)); };
        hipError_t e = hipSuccess;
        if (OUT) {
            for (size_t k = 0; k < std::min<size_t>(2, pieces) && e == hipSuccess; ++k) e = issue(at(k), len(k), slots + (k & 1) * slot, ev[k & 1]);
            for (size_t k = 0; k < pieces && e == hipSuccess; ++k) {
                if ((e = hipEventSynchronize(ev[k & 1])) != hipSuccess) break;
                host_copy(at(k), len(k), slots + (k & 1) * slot);
                if (k + 2 < pieces) e = issue(at(k + 2), len(k + 2), slots + (k & 1) * slot, ev[k & 1]);
            }
        } else {
            for (size_t k = 0; k < pieces && e == hipSuccess; ++k) {
                if (k >= 2 && (e = hipEventSynchronize(ev[k & 1])) != hipSuccess) break;
                host_copy(at(k), len(k), slots + (k & 1) * slot);
                e = issue(at(k), len(k), slots + (k & 1) * slot, ev[k & 1]);
            }
            for (size_t k = pieces > 2 ? pieces - 2 : 0; k < pieces && e == hipSuccess; ++k) e = hipEventSynchronize(ev[k & 1]);
        }
        if (e != hipSuccess) (void)hipStreamSynchronize(s);
        return e;
    }
};

template <class H, bool OUT>
hipError_t transfer(HostStage &st, int device, hipStream_t s, const XferArray *arrays, int n) {
    Transfer<H, OUT> x = {s, arrays, n, {}, 0};
    unsigned long long total = 0;
    for (int k = 0; k < kMaxArrays; ++k) {
        x.lay.begin[k] = total;
        if (k < n) {
            x.lay.dev[k] = arrays[k].dev;
            x.lay.layout[k] = arrays[k].layout;
            x.lay.wide[k] = arrays[k].wide;
            total += arrays[k].count;
        }
    }
    x.lay.begin[kMaxArrays] = total;
    const OnDevice here(device);
    if (total == 0) return hipStreamSynchronize(s);
    const size_t bytes = (size_t)total * sizeof(H);
    const int threads = bytes >= kXferLarge ? kXferThreads : 1;
    // A small owner keeps small slots.  Below kXferWhole one piece is quicker than two that overlap.
    const size_t slot = std::min(kXferSlot, ((bytes < kXferWhole ? bytes : bytes / 2) + 4095) / 4096 * 4096);
    const size_t need = 2 * slot * threads;
    x.slot = slot / sizeof(H);
    hipError_t e;
    if (st.bytes < need) {
        if (st.pin) (void)hipHostFree(st.pin);
        st.pin = nullptr;
        st.bytes = 0;
        if ((e = hipHostMalloc((void **)&st.pin, need, 0)) != hipSuccess) return e;
        st.bytes = need;
    }
    for (int k = 0; k < 2 * threads; ++k)
        if (!st.ev[k] && (e = hipEventCreateWithFlags(&st.ev[k], hipEventDisableTiming)) != hipSuccess) return e;
    hipError_t res[kXferThreads] = {};
    const size_t per = ((size_t)total + threads - 1) / threads;
    auto part = [&](int t) {
        const size_t lo = std::min((size_t)total, per * t), hi = std::min((size_t)total, lo + per);
        res[t] = x.part(lo, hi, (H *)(st.pin + 2 * slot * t), st.ev + 2 * t);
    };
    std::vector<std::thread> pool;
    int started = 1;
    try {
        for (; started < threads; ++started)
            pool.emplace_back([&, t = started] {
                if ((res[t] = hipSetDevice(device)) == hipSuccess) part(t);
            });
    } catch (...) {  // no further thread to be had: this one does the rest
    }
    part(0);
    for (int t = started; t < threads; ++t) part(t);
    for (std::thread &t : pool) t.join();
    for (int t = 0; t < threads; ++t)
        if (res[t] != hipSuccess) return res[t];
    return hipSuccess;
}

template <class H>
int state_arrays(XferArray *x, size_t n, bool wide, const void *pos, const void *vel, const void *acc, H *r, H *v, H *a) {
    int k = 0;
    if (r) x[k++] = {(void *)r, pos, 4 * n, XferLayout::plain, wide};
    if (v) x[k++] = {(void *)v, vel, 3 * n, XferLayout::blocks, wide};
    if (a) x[k++] = {(void *)a, acc, 3 * n, XferLayout::blocks, wide};
    return k;
}

}  // namespace

void stage_free(HostStage &st) {
    if (st.pin) (void)hipHostFree(st.pin);
    for (hipEvent_t e : st.ev)
        if (e) (void)hipEventDestroy(e);
    st = {};
}

template <class H>
hipError_t xfer_to_host(HostStage &st, int device, hipStream_t s, const XferArray *arrays, int n) {
    return transfer<H, true>(st, device, s, arrays, n);
}

template <class H>
hipError_t state_to_host(HostStage &st, int device, hipStream_t s, size_t n, bool wide, const void *pos, const void *vel,
                         const void *acc, H *r, H *v, H *a) {
    XferArray x[kMaxArrays];
    return transfer<H, true>(st, device, s, x, state_arrays(x, n, wide, pos, vel, acc, r, v, a));
}
template <class H>
hipError_t state_to_device(HostStage &st, int device, hipStream_t s, size_t n, bool wide, const H *r, const H *v,
                           const H *a, void *pos, void *vel, void *acc) {
    XferArray x[kMaxArrays];
    return transfer<H, false>(st, device, s, x, state_arrays(x, n, wide, pos, vel, acc, r, v, a));
}

#define SGK_XFER(H)                                                                                                    \
    template hipError_t xfer_to_host<H>(HostStage &, int, hipStream_t, const XferArray *, int);                       \
    template hipError_t state_to_host<H>(HostStage &, int, hipStream_t, size_t, bool, const void *, const void *,     \
                                         const void *, H *, H *, H *);                                                \
    template hipError_t state_to_device<H>(HostStage &, int, hipStream_t, size_t, bool, const H *, const H *,         \
                                           const H *, void *, void *, void *);
SGK_XFER(double)
SGK_XFER(float)
#undef SGK_XFER

}  // namespace sgk
