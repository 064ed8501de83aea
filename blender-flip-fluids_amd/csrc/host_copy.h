// host_copy.h -- device data into a caller's pageable memory.
//
// What bounds it: the first touch of the caller's pages.  A fresh 45 MB buffer
// takes 10 ms of page faults on one thread (a copy into pages that are there
// 1.4 ms), the link 0.8 ms.  So a kernel writes the data in its final layout
// straight to pinned memory (54 GB/s, what a plain device-to-host copy
// reaches), in halves, and several threads copy one half out while the next
// is on its way: 2.0 ms with eight threads.  Three copies into pageable
// memory and an interleaving loop on the host took 25 ms.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <stdexcept>
#include <system_error>
#include <thread>
#include <vector>

#include <hip/hip_runtime_api.h>

namespace ff {

void hipCheck(hipError_t e, const char *what);

class HostCopy {
public:
    HostCopy() = default;
    HostCopy(const HostCopy &) = delete;
    HostCopy &operator=(const HostCopy &) = delete;
    ~HostCopy() {
        if (_pinned) (void)hipHostFree(_pinned);
    }
    // out receives `bytes` bytes.  fill(dst, lo, n) enqueues on s what writes
    // bytes [lo, lo + n) of the data to the pinned dst; lo is a multiple of
    // HALF.  All of them are in out on return.  Several threads may call it at
    // once (one reads positions, another velocities): they share the pinned
    // buffer and take turns, as their copies would on the link.
    template <class Fill>
    void run(char *out, size_t bytes, hipStream_t s, Fill fill) {
        if (bytes == 0) return;
        if (!out) throw std::domain_error("Error: no buffer to read back into.\n");
        std::lock_guard<std::mutex> turn(_turn);
        const OnDevice on(s);
        reserve(bytes);
        const int halves = (int)((bytes + HALF - 1) / HALF);
        // a thread's start costs about as much as 256 KB of copying
        const unsigned cores = std::thread::hardware_concurrency();
        const size_t most = cores > 8 ? 8 : cores > 1 ? cores : 1;
        const size_t want = std::min(most, bytes / (1 << 20) + 1);
        const auto slice = [&](int h, size_t part, size_t parts) {
            const size_t lo = (size_t)h * HALF, n = std::min(HALF, bytes - lo);
            const size_t step = ((n + parts - 1) / parts + 4095) / 4096 * 4096;
            const size_t a = std::min(part * step, n), b = std::min(a + step, n);
            memcpy(out + lo + a, half(h) + a, b - a);
        };
        Team team;  // after what its threads use
        fill(half(0), (size_t)0, std::min(HALF, bytes));
        team.start(want - 1, halves, slice);
        for (int h = 0; h < halves; h++) {
            hipCheck(hipStreamSynchronize(s), "read-back");
            team.awaitDone(h);  // the other half is free again
            if (h + 1 < halves) {
                const size_t lo = (size_t)(h + 1) * HALF;
                fill(half(h + 1), lo, std::min(HALF, bytes - lo));
            }
            team.release(h + 1);
            slice(h, 0, team.size() + 1);
        }
        team.awaitDone(halves);
    }
    // `bytes` contiguous bytes at the device address src
    void run(char *out, const void *src, size_t bytes, hipStream_t s) {
        run(out, bytes, s, [&](char *dst, size_t lo, size_t n) {
            hipCheck(hipMemcpyAsync(dst, (const char *)src + lo, n, hipMemcpyDeviceToHost, s), "read-back");
        });
    }

    // a multiple of 12 (three floats) and of 16
    static constexpr size_t HALF = (size_t)48 * 350000;

private:
    // The calling thread is on the stream's device for a while: fill launches a
    // kernel, and a thread that has chosen no device is on device 0.
    class OnDevice {
    public:
        explicit OnDevice(hipStream_t s) {
            int device = 0;
            hipCheck(hipGetDevice(&_before), "hipGetDevice");
            hipCheck(hipStreamGetDevice(s, &device), "hipStreamGetDevice");
            if (device == _before) return;
            hipCheck(hipSetDevice(device), "hipSetDevice");
            _changed = true;
        }
        ~OnDevice() {
            if (_changed) (void)hipSetDevice(_before);
        }
        OnDevice(const OnDevice &) = delete;
        OnDevice &operator=(const OnDevice &) = delete;

    private:
        int _before = 0;
        bool _changed = false;
    };

    // The helper threads of one call.  Half h may be copied once released > h;
    // the destructor ends and joins them whatever happened.
    class Team {
    public:
        ~Team() {
            {
                std::lock_guard<std::mutex> l(_m);
                _stop = true;
            }
            _cv.notify_all();
            for (auto &t : _threads) t.join();
        }
        template <class Slice>
        void start(size_t helpers, int halves, const Slice &slice) {
            _threads.reserve(helpers);
            try {
                for (size_t q = 0; q < helpers; q++)
                    _threads.emplace_back([this, halves, &slice, part = q + 1] {
                        for (int h = 0; h < halves; h++) {
                            size_t parts;
                            {
                                std::unique_lock<std::mutex> l(_m);
                                _cv.wait(l, [&] { return _stop || _released > h; });
                                if (_released <= h) return;
                                parts = _threads.size() + 1;  // all are started before the first release
                            }
                            slice(h, part, parts);
                            {
                                std::lock_guard<std::mutex> l(_m);
                                _done++;
                            }
                            _cv.notify_all();
                        }
                    });
            } catch (const std::system_error &) {
                // no more threads to be had: the ones there are share the work
            }
        }
        size_t size() const { return _threads.size(); }
        void release(int halves) {
            {
                std::lock_guard<std::mutex> l(_m);
                _released = halves;
            }
            _cv.notify_all();
        }
        void awaitDone(int halves) {
            std::unique_lock<std::mutex> l(_m);
            _cv.wait(l, [&] { return _done >= halves * (int)_threads.size(); });
        }

    private:
        std::vector<std::thread> _threads;
        std::mutex _m;
        std::condition_variable _cv;
        int _released = 0, _done = 0;
        bool _stop = false;
    };

    char *half(int h) { return _pinned + (h & 1 ? HALF : 0); }
    void reserve(size_t bytes) {
        const size_t need = std::min(bytes, 2 * HALF);
        if (need <= _size) return;
        if (_pinned) hipCheck(hipHostFree(_pinned), "read-back buffer");
        _pinned = nullptr;
        _size = 0;
        hipCheck(hipHostMalloc((void **)&_pinned, need, hipHostMallocDefault), "read-back buffer");
        _size = need;
    }
    std::mutex _turn;
    char *_pinned = nullptr;
    size_t _size = 0;
};

}  // namespace ff
