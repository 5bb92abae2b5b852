#include "hostcopy.h"

#include <cstring>

#include "runtime.h"

namespace zjai {

namespace {

bool page_locked(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();  // not an error of the caller's: ordinary memory
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

}  // namespace

void HostCopier::create() {
    void* p = nullptr;
    ZJAI_HIP(hipHostMalloc(&p, SLOT * SLOTS, hipHostMallocDefault));
    slots_ = (char*)p;
    for (hipEvent_t& e : ev_) ZJAI_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    ZJAI_HIP(hipEventCreateWithFlags(&order_, hipEventDisableTiming));
    ZJAI_HIP(hipStreamCreateWithFlags(&side_, hipStreamNonBlocking));
}

HostCopier::~HostCopier() {
    for (int i = 0; i < SLOTS; ++i)
        if (pending_[i]) (void)hipEventSynchronize(ev_[i]);
    if (side_) {
        (void)hipStreamSynchronize(side_);
        (void)hipStreamDestroy(side_);
    }
    for (hipEvent_t e : ev_)
        if (e) (void)hipEventDestroy(e);
    if (order_) (void)hipEventDestroy(order_);
    if (slots_) (void)hipHostFree(slots_);
}

void HostCopier::order(hipStream_t first, hipStream_t later) {
    ZJAI_HIP(hipEventRecord(order_, first));
    ZJAI_HIP(hipStreamWaitEvent(later, order_, 0));
}

int HostCopier::take() {
    const int k = next_;
    next_ = (next_ + 1) % SLOTS;
    if (pending_[k]) ZJAI_HIP(hipEventSynchronize(ev_[k]));
    pending_[k] = false;
    return k;
}

void HostCopier::to_device(void* dst, const void* src, size_t n, hipStream_t s) {
    if (!slots_ || n == 0 || n > SLOT || page_locked(src)) {
        ZJAI_HIP(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, s));
        return;
    }
    const int k = take();
    std::memcpy(slot(k), src, n);
    pending_[k] = true;  // before the copy: an error after it must not free the slot early
    ZJAI_HIP(hipMemcpyAsync(dst, slot(k), n, hipMemcpyHostToDevice, s));
    ZJAI_HIP(hipEventRecord(ev_[k], s));
}

void HostCopier::to_host(void* dst, const void* src, size_t n, hipStream_t s) {
    if (!slots_ || n == 0 || n > SLOT || page_locked(dst)) {
        ZJAI_HIP(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, s));
        return;
    }
    const int k = take();
    ZJAI_HIP(hipMemcpyAsync(slot(k), src, n, hipMemcpyDeviceToHost, s));
    ZJAI_HIP(hipStreamSynchronize(s));
    std::memcpy(dst, slot(k), n);
}

}  // namespace zjai
