// Copies between a caller's dense host array and a padded device array.
//
// A two-dimensional copy call moves such an array row by row, 8 us a row
// whatever its length (8.1 ms for 1028 rows of 8 KB). Here a kernel gathers
// the rows straight into pinned host memory, or scatters them from it, over
// PCIe (50 GB/s), a chunk at a time, while the host copies the chunks before
// it to or from the caller's array: 0.34 ms for the same array, bound by the
// host's own copy into fresh pages.
#ifndef INCRMT_HOSTCOPY_HH
#define INCRMT_HOSTCOPY_HH

#include <cstring>
#include "common.hh"

namespace incrmt {

// count host elements from element (i0, j0) of the dense w-wide array: the
// device array's columns past wd read as zero and are not written
template <class D, class H>
__global__ void k_rows_to_host(const D *dev, long long pitch, int w, int wd, int i0, long long j0, int count, H *host) {
    const unsigned k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (unsigned)count) return;
    const unsigned r = ((unsigned)i0 + k) / (unsigned)w, i = (unsigned)i0 + k - r * (unsigned)w;
    host[k] = i < (unsigned)wd ? (H)dev[(j0 + r) * pitch + i] : (H)0;
}
template <class D, class H>
__global__ void k_rows_from_host(D *dev, long long pitch, int w, int wd, int i0, long long j0, int count, const H *host) {
    const unsigned k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (unsigned)count) return;
    const unsigned r = ((unsigned)i0 + k) / (unsigned)w, i = (unsigned)i0 + k - r * (unsigned)w;
    if (i < (unsigned)wd) dev[(j0 + r) * pitch + i] = (D)host[k];
}

// One handle's pinned chunks, allocated by its first copy (no more than that
// array needs, 4 MiB at most) and kept for the next; copies wait for their
// stream, as the handle's other calls do.
class HostCopy {
  public:
    ~HostCopy() {
        if (pin_) (void)hipHostFree(pin_);
        for (hipEvent_t e : ev_)
            if (e) (void)hipEventDestroy(e);
    }
    // h rows of w host elements; the device rows hold wd <= w of them
    template <class D, class H>
    int down(hipStream_t s, const D *dev, long long pitch, int w, int wd, long long h, H *host) {
        const long long n = (long long)w * h;
        if (int rc = reserve(n * (long long)sizeof(H))) return rc;
        const long long per = chunk_ / (long long)sizeof(H), chunks = (n + per - 1) / per;
        auto ask = [&](long long c) -> int {
            const long long e0 = c * per, cnt = n - e0 < per ? n - e0 : per;
            k_rows_to_host<D, H><<<(unsigned)((cnt + 255) / 256), 256, 0, s>>>(
                dev, pitch, w, wd, (int)(e0 % w), e0 / w, (int)cnt, (H *)(pin_ + c % slots_ * chunk_));
            HIP_CHECK(hipGetLastError());
            HIP_CHECK(hipEventRecord(ev_[c % slots_], s));
            return 0;
        };
        long long asked = 0;
        for (; asked < chunks && asked < slots_; asked++)
            if (int rc = ask(asked)) return rc;
        for (long long c = 0; c < chunks; c++) {
            HIP_CHECK(hipEventSynchronize(ev_[c % slots_]));
            const long long e0 = c * per, cnt = n - e0 < per ? n - e0 : per;
            std::memcpy(host + e0, pin_ + c % slots_ * chunk_, (size_t)cnt * sizeof(H));
            if (asked < chunks)
                if (int rc = ask(asked++)) return rc;
        }
        return 0;
    }
    template <class D, class H>
    int up(hipStream_t s, D *dev, long long pitch, int w, int wd, long long h, const H *host) {
        const long long n = (long long)w * h;
        if (int rc = reserve(n * (long long)sizeof(H))) return rc;
        const long long per = chunk_ / (long long)sizeof(H), chunks = (n + per - 1) / per;
        for (long long c = 0; c < chunks; c++) {
            const long long e0 = c * per, cnt = n - e0 < per ? n - e0 : per;
            if (c >= slots_) HIP_CHECK(hipEventSynchronize(ev_[c % slots_]));  // the slot's last reader
            std::memcpy(pin_ + c % slots_ * chunk_, host + e0, (size_t)cnt * sizeof(H));
            k_rows_from_host<D, H><<<(unsigned)((cnt + 255) / 256), 256, 0, s>>>(
                dev, pitch, w, wd, (int)(e0 % w), e0 / w, (int)cnt, (const H *)(pin_ + c % slots_ * chunk_));
            HIP_CHECK(hipGetLastError());
            HIP_CHECK(hipEventRecord(ev_[c % slots_], s));
        }
        HIP_CHECK(hipStreamSynchronize(s));
        return 0;
    }

  private:
    static constexpr int kSlots = 4;
    static constexpr long long kChunk = 1 << 20;
    char *pin_ = nullptr;
    long long chunk_ = 0;
    int slots_ = 0;
    hipEvent_t ev_[kSlots] = {nullptr, nullptr, nullptr, nullptr};
    int reserve(long long bytes) {
        const long long chunk = bytes < kChunk ? (bytes + 255) / 256 * 256 : kChunk;
        const int slots = (int)(bytes / chunk + (bytes % chunk != 0) < kSlots ? bytes / chunk + (bytes % chunk != 0) : kSlots);
        for (int k = 0; k < slots; k++)
            if (!ev_[k]) HIP_CHECK(hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming));
        if (pin_ && chunk <= chunk_ && slots <= slots_) return 0;
        if (pin_) HIP_CHECK(hipHostFree(pin_));
        pin_ = nullptr;
        HIP_CHECK(hipHostMalloc((void **)&pin_, (size_t)(chunk * slots), hipHostMallocDefault));
        chunk_ = chunk;
        slots_ = slots;
        return 0;
    }
};

}  // namespace incrmt

#endif
