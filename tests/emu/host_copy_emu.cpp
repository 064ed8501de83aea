// host_copy_emu.cpp -- the read-back's host side
// (blender-flip-fluids_amd/csrc/host_copy.h) with the HIP calls it makes
// replaced by plain memory: device memory is host memory, pinned memory is
// malloc's, and a copy lands when its stream is waited for.
//
// Usage: host_copy_emu <threads>
// Each thread reads its own arrays back through one HostCopy, of sizes around
// its halves, ascending (so the pinned buffer is replaced under way), and
// compares every byte; the copies are made on the stream's device, which is not
// the threads' own.  Exit status 0: all equal.  Built with a sanitizer.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <stdexcept>

#include "../../blender-flip-fluids_amd/csrc/host_copy.h"

namespace ff {
void hipCheck(hipError_t e, const char *what) {
    if (e != hipSuccess) throw std::runtime_error(what);
}
}  // namespace ff

static std::mutex gM;
static std::vector<std::function<void()>> gQueue;  // the one stream's work

constexpr int STREAM_DEVICE = 3;
static thread_local int gDevice = 0;
static std::atomic<int> gElsewhere{0};  // copies asked for on another device

extern "C" hipError_t hipGetDevice(int *d) {
    *d = gDevice;
    return hipSuccess;
}
extern "C" hipError_t hipSetDevice(int d) {
    gDevice = d;
    return hipSuccess;
}
extern "C" hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) {
    *d = STREAM_DEVICE;
    return hipSuccess;
}
extern "C" hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::malloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
extern "C" hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
extern "C" hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
    if (gDevice != STREAM_DEVICE) gElsewhere++;
    std::lock_guard<std::mutex> l(gM);
    gQueue.push_back([=] { std::memcpy(dst, src, n); });
    return hipSuccess;
}
extern "C" hipError_t hipStreamSynchronize(hipStream_t) {
    std::this_thread::sleep_for(std::chrono::milliseconds(1));
    std::lock_guard<std::mutex> l(gM);
    for (auto &f : gQueue) f();
    gQueue.clear();
    return hipSuccess;
}

int main(int argc, char **argv) {
    if (argc != 2) return 2;
    const int threads = std::atoi(argv[1]);
    constexpr size_t H = ff::HostCopy::HALF;
    ff::HostCopy copy;
    std::atomic<int> bad{0};
    try {  // no destination: an error, and nothing written
        copy.run(nullptr, &copy, 1, nullptr);
        bad++;
    } catch (const std::domain_error &) {
    }
    std::vector<std::thread> team;
    for (int t = 0; t < threads; t++)
        team.emplace_back([&, t] {
            for (size_t bytes : {(size_t)0, (size_t)1, (size_t)4097, (size_t)3 << 20, H - 1, H, H + 1, 2 * H + 5}) {
                std::vector<char> from(bytes), to(bytes + 2, 'x');
                for (size_t q = 0; q < bytes; q++) from[q] = (char)((q * 2654435761u >> 13) + 31 * t);
                copy.run(to.data() + 1, from.data(), bytes, nullptr);  // an odd address
                if (to[0] != 'x' || to[bytes + 1] != 'x' || (bytes && std::memcmp(to.data() + 1, from.data(), bytes))) bad++;
                if (gDevice != 0) bad++;
            }
        });
    for (auto &t : team) t.join();
    if (bad) std::fprintf(stderr, "host_copy_emu: %d read-backs differ\n", (int)bad);
    if (gElsewhere) std::fprintf(stderr, "host_copy_emu: %d copies on another device\n", (int)gElsewhere);
    return bad || gElsewhere ? 1 : 0;
}
