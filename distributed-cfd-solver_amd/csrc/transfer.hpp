// Copies between a caller's pageable host array and device memory.
//
// A pageable hipMemcpy moves a large array through the runtime's staging buffer
// with one thread that alternates between its host copy and the device copy.
// Here up to eight threads each move pieces of 1 MiB through two pinned slots of
// their own, so the host copies run side by side (and fault in the pages of a
// freshly allocated array side by side) while the device copies of other pieces
// are in flight.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace cfdg {

class HostPipe {
  public:
    HostPipe() = default;
    HostPipe(const HostPipe&) = delete;
    HostPipe& operator=(const HostPipe&) = delete;
    ~HostPipe();
    // Pinned slots for arrays of up to this many bytes on the current device;
    // none are made when all are small, and without pinned memory for them every array
    // goes through the runtime's copy.
    void reserve(std::size_t bytes);
    // The copies run on s after the work already enqueued there.  to_device's source stays
    // as it is until s is waited for (small arrays are read by then, others on return);
    // to_host returns with the array written.
    void to_device(void* dst, const void* src, std::size_t bytes, hipStream_t s);
    void to_host(void* dst, const void* src, std::size_t bytes, hipStream_t s);

  private:
    static constexpr int kWorkers = 8, kSlots = 2 * kWorkers;
    static constexpr std::size_t kPiece = 1u << 20;
    // below this one runtime copy is as fast as starting the threads
    static constexpr std::size_t kSmall = 2 * kPiece;
    template <class F>
    void run(std::size_t bytes, F&& worker);
    bool piped(std::size_t bytes) const { return pinned_ && bytes >= kSmall; }

    char* pinned_ = nullptr;
    hipEvent_t ev_[kSlots] = {};
    int device_ = 0;
};

}  // namespace cfdg
