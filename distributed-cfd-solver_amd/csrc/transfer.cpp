// Pipelined host <-> device copies (transfer.hpp).
#include "transfer.hpp"

#include <algorithm>
#include <cstring>
#include <exception>
#include <string>
#include <thread>
#include <vector>

#include "capi_internal.hpp"
#include "cfdg.h"

namespace cfdg {

namespace {

inline std::size_t z(int v) { return static_cast<std::size_t>(v); }

void check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw CfdgError(CFDG_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

}  // namespace

HostPipe::~HostPipe() {
    for (hipEvent_t e : ev_)
        if (e) (void)hipEventDestroy(e);
    if (pinned_) (void)hipHostFree(pinned_);
}

void HostPipe::reserve(std::size_t bytes) {
    if (pinned_ || bytes < kSmall) return;
    check(hipGetDevice(&device_), "hipGetDevice");
    for (hipEvent_t& e : ev_)
        if (!e) check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
    if (hipHostMalloc(reinterpret_cast<void**>(&pinned_), kSlots * kPiece) != hipSuccess) {
        pinned_ = nullptr;
        (void)hipGetLastError();  // the runtime's own copies do without
    }
}

// worker(w, workers) on every thread; the first error is thrown when all have
// ended.  Pieces w, w + workers, ... belong to worker w and alternate between
// its two slots.  Threads that cannot be started leave their pieces to fewer.
template <class F>
void HostPipe::run(std::size_t bytes, F&& worker) {
    const std::size_t pieces = (bytes + kPiece - 1) / kPiece;
    const int want = static_cast<int>(std::min<std::size_t>(kWorkers, (pieces + 1) / 2));
    hipError_t err[kWorkers] = {};
    std::vector<std::thread> th;
    th.reserve(kWorkers);
    int started = 0;
    const auto body = [&](int w) {
        err[w] = hipSetDevice(device_);
        if (err[w] == hipSuccess) err[w] = worker(w, want);
    };
    try {
        for (; started + 1 < want; ++started) th.emplace_back(body, started + 1);
    } catch (const std::exception&) {  // no thread, or no memory for one
    }
    body(0);
    for (int w = started + 1; w < want; ++w) body(w);
    for (std::thread& t : th) t.join();
    for (hipError_t e : err) check(e, "host copy");
}

void HostPipe::to_device(void* dst, const void* src, std::size_t bytes, hipStream_t s) {
    if (bytes == 0) return;
    if (!piped(bytes)) {
        check(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s), "H2D");
        return;
    }
    run(bytes, [&](int w, int workers) -> hipError_t {
        int k = 0;
        for (std::size_t at = z(w) * kPiece; at < bytes; at += z(workers) * kPiece, ++k) {
            const int slot = 2 * w + (k & 1);
            const std::size_t n = std::min(kPiece, bytes - at);
            char* const buf = pinned_ + z(slot) * kPiece;
            // the slot's last copy, of this call or an earlier one
            hipError_t e = hipEventSynchronize(ev_[slot]);
            if (e != hipSuccess) return e;
            std::memcpy(buf, static_cast<const char*>(src) + at, n);
            e = hipMemcpyAsync(static_cast<char*>(dst) + at, buf, n, hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(ev_[slot], s);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    });
}

void HostPipe::to_host(void* dst, const void* src, std::size_t bytes, hipStream_t s) {
    if (bytes == 0) return;
    if (!piped(bytes)) {
        check(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s), "D2H");
        check(hipStreamSynchronize(s), "hipStreamSynchronize");
        return;
    }
    run(bytes, [&](int w, int workers) -> hipError_t {
        const std::size_t step = z(workers) * kPiece;
        const auto fetch = [&](std::size_t at, int slot) -> hipError_t {
            const hipError_t e = hipMemcpyAsync(pinned_ + z(slot) * kPiece, static_cast<const char*>(src) + at,
                                                std::min(kPiece, bytes - at), hipMemcpyDeviceToHost, s);
            return e == hipSuccess ? hipEventRecord(ev_[slot], s) : e;
        };
        const std::size_t first = z(w) * kPiece;
        for (int k = 0; k < 2 && first + z(k) * step < bytes; ++k) {
            // an earlier to_device may still read the slot: same stream, so the copy waits for it
            const hipError_t e = fetch(first + z(k) * step, 2 * w + k);
            if (e != hipSuccess) return e;
        }
        int k = 0;
        for (std::size_t at = first; at < bytes; at += step, ++k) {
            const int slot = 2 * w + (k & 1);
            hipError_t e = hipEventSynchronize(ev_[slot]);
            if (e != hipSuccess) return e;
            std::memcpy(static_cast<char*>(dst) + at, pinned_ + z(slot) * kPiece, std::min(kPiece, bytes - at));
            if (at + 2 * step < bytes && (e = fetch(at + 2 * step, slot)) != hipSuccess) return e;
        }
        return hipSuccess;
    });
}

}  // namespace cfdg
