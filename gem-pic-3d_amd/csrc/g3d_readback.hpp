// Copies of large device arrays to ordinary host memory.
#pragma once
#include <algorithm>
#include <cstring>
#include <stdexcept>
#include <thread>
#include <vector>
#include "g3d_runtime.hpp"

namespace g3d {

// A large array to ordinary host memory: kReaders threads, each with two pinned buffers on the library's stream, copy one
// chunk out while the next arrives.  The runtime's own copy to memory that is not pinned is serial and takes the page
// faults of a new array in one thread: 409 MB 38 -> 13 ms, 102 MB 9.7 -> 3.3, 51 MB 4.9 -> 1.8; at 34 MB 3.1 ms against
// 1.4 to 3.8, hence kReadMin.  The buffers (32 MB) live for the call.  False when they or the threads are not to be had;
// then nothing has been copied that a plain copy would not write again.
constexpr size_t kReadChunk = size_t(2) << 20, kReadMin = size_t(48) << 20;
constexpr int kReaders = 8;
inline bool read_staged(char* host, const char* dev, size_t bytes) {
    struct Staging {
        char* pin = nullptr;
        hipEvent_t ev[2 * kReaders] = {};
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;       // another thread may be capturing a graph
        bool swapped = false;
        ~Staging() {
            if (pin) (void)hipStreamSynchronize(stream());
            for (auto e : ev) if (e) (void)hipEventDestroy(e);
            if (pin) (void)hipHostFree(pin);
            if (swapped) (void)hipThreadExchangeStreamCaptureMode(&mode);
        }
    };
    struct Joined {
        std::vector<std::thread> t;
        ~Joined() { for (auto& x : t) x.join(); }
    };
    hipError_t err[kReaders] = {};
    {
        Staging g;
        int device = 0;
        g.swapped = hipThreadExchangeStreamCaptureMode(&g.mode) == hipSuccess;
        if (!g.swapped || hipGetDevice(&device) != hipSuccess ||
            hipHostMalloc(reinterpret_cast<void**>(&g.pin), 2 * kReaders * kReadChunk, hipHostMallocDefault) != hipSuccess) {
            g.pin = nullptr;
            (void)hipGetLastError();
            return false;
        }
        for (auto& e : g.ev)
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) { e = nullptr; (void)hipGetLastError(); return false; }
        const size_t n = (bytes + kReadChunk - 1) / kReadChunk;
        auto reader = [&](int r) {
            hipError_t& rc = err[r];
            char* buf[2] = {g.pin + 2 * r * kReadChunk, g.pin + (2 * r + 1) * kReadChunk};
            auto size = [&](size_t c) { return std::min(kReadChunk, bytes - c * kReadChunk); };
            auto fetch = [&](size_t c, int b) {
                if (c >= n || rc != hipSuccess) return;
                rc = hipMemcpyAsync(buf[b], dev + c * kReadChunk, size(c), hipMemcpyDeviceToHost, stream());
                if (rc == hipSuccess) rc = hipEventRecord(g.ev[2 * r + b], stream());
            };
            rc = hipSetDevice(device);
            int b = 0;
            fetch(r, 0);
            for (size_t c = r; c < n && rc == hipSuccess; c += kReaders, b ^= 1) {
                fetch(c + kReaders, b ^ 1);
                if (rc == hipSuccess) rc = hipEventSynchronize(g.ev[2 * r + b]);
                if (rc == hipSuccess) std::memcpy(host + c * kReadChunk, buf[b], size(c));
            }
        };
        Joined j;                        // after all that the threads refer to: joined before any of it goes out of scope
        try {
            j.t.reserve(kReaders);
            for (int r = 0; r < kReaders; ++r) j.t.emplace_back(reader, r);
        } catch (const std::exception&) { return false; }
    }
    for (const hipError_t e : err) hip_check(e, "hipMemcpy D2H");
    return true;
}

}  // namespace g3d
