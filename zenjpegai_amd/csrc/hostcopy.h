// Copies between device memory and the caller's ordinary (pageable) host memory.
#pragma once

#include <hip/hip_runtime.h>

namespace zjai {

// A copy of up to SLOT bytes goes through a page-locked slot; a larger one is left to the runtime's
// staging. The runtime takes ~10 us of set-up per pageable copy whatever its size, which a call on a
// 64x96 tile pays three times in ~150 us; at 1 MB its own two-buffer staging was as fast as a slot.
//
// One per context, used by one thread at a time, as the context is.
class HostCopier {
public:
    static constexpr size_t SLOT = 256u << 10;
    static constexpr int SLOTS = 4;
    void create();
    // In stream order on the device. A pageable `src` may be reused on return; a page-locked one is read in
    // stream order too, and stays until `s` has got there.
    void to_device(void* dst, const void* src, size_t n, hipStream_t s);
    // Page-locked `dst`: in stream order. Pageable `dst`: holds the bytes on return.
    void to_host(void* dst, const void* src, size_t n, hipStream_t s);
    // A second stream for downloads that need not wait for later work.
    hipStream_t side_stream() const { return side_; }
    // Work put into `later` from here on runs after what `first` holds now.
    void order(hipStream_t first, hipStream_t later);
    HostCopier() = default;
    HostCopier(const HostCopier&) = delete;
    HostCopier& operator=(const HostCopier&) = delete;
    ~HostCopier();

private:
    int take();
    char* slot(int k) { return slots_ + (size_t)k * SLOT; }

    char* slots_ = nullptr;
    hipEvent_t ev_[SLOTS] = {};
    bool pending_[SLOTS] = {};  // the slot's last upload may still be reading it
    int next_ = 0;
    hipStream_t side_ = nullptr;
    hipEvent_t order_ = nullptr;
};

}  // namespace zjai
