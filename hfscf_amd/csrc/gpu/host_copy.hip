// Copy of a large device vector to pageable host memory.
//
// One hipMemcpy into pages the caller has not touched yet is bound by one host thread that faults them
// in and copies: 10 GB/s, where the link gives 52. Here up to kThreads host threads take chunks in turn; each
// has the device write a chunk into one of its two pinned buffers while it copies the other one out, so that
// the page faults and the copies of the threads run beside the link's transfers. Measured on 1.6 GB,
// fresh huge / small pages: one thread 117 / 349 ms, 2 61 / 214, 4 39 / 122,
// 8 35 / 71, 12 35 / 61; chunks of 1 MB 51 ms, 4 MB 35, 16 MB 31 but 88 on small pages. The buffers live
// for the call only. Pinned memory that the runtime does not hold from before costs about 70 us per MB (its first
// use above all), so the chunks are a 32nd of the vector where that is less than 4 MB: with 4 MB (64 MB of buffers)
// the 32 MB vector of (H2O)3 / 6-31G** took 6.5 ms with its kernels, as long as the plain copy, now 2.1; 87 MB 11.8 ->
// 6.1, 172 MB 9.7 -> 5.4. The 1.37 GB vector of (H2O)8 / cc-pVDZ: 145 ms with the plain copy, 38 so.
#include "host_copy.hpp"

#include <algorithm>
#include <array>
#include <atomic>
#include <cstring>
#include <thread>

namespace hfg {

namespace {
constexpr size_t kMinChunk = 1 << 20, kMaxChunk = 4 << 20;  // whole MB between them
constexpr int kThreads = 8;
// Below this the plain copy: the threads and buffers cost 0.1 ms. Plain / staged into touched pages: 4 MB
// 0.24 / 0.29 ms, 8 MB 0.47 / 0.44, 16 MB 0.94 / 0.62, 64 MB 3.8 / 1.7.
constexpr size_t kStagedBytes = 16 << 20;
}  // namespace

hipError_t copy_to_host(void* dst, const void* src, size_t bytes, int device, hipStream_t st) {
    const size_t chunk = std::min(kMaxChunk, std::max(kMinChunk, bytes / 32 / kMinChunk * kMinChunk));
    const size_t nchunk = (bytes + chunk - 1) / chunk;
    const int want = (int)std::min<size_t>({(size_t)kThreads, std::max(1u, std::thread::hardware_concurrency()), nchunk});
    char* pinned = nullptr;
    if (bytes < kStagedBytes || hipHostMalloc((void**)&pinned, 2 * want * chunk, 0) != hipSuccess) {
        (void)hipGetLastError();
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
        return e != hipSuccess ? e : hipStreamSynchronize(st);
    }
    std::atomic<size_t> next{0};
    std::atomic<int> error{hipSuccess};
    auto work = [&](int t) {
        hipEvent_t ev[2] = {nullptr, nullptr};
        size_t held[2] = {nchunk, nchunk};  // the chunk in flight to each buffer
        auto check = [&](hipError_t e) {
            if (e != hipSuccess) error = (int)e;
            return e == hipSuccess && error == hipSuccess;
        };
        auto issue = [&](int s) {
            held[s] = next.fetch_add(1);
            if (held[s] >= nchunk) return true;
            const size_t off = held[s] * chunk;
            return check(hipMemcpyAsync(pinned + (2 * (size_t)t + s) * chunk, (const char*)src + off,
                                        std::min(chunk, bytes - off), hipMemcpyDeviceToHost, st)) &&
                   check(hipEventRecord(ev[s], st));
        };
        bool ok = check(hipSetDevice(device));
        for (int s = 0; s < 2 && ok; ++s) ok = check(hipEventCreateWithFlags(&ev[s], hipEventDisableTiming));
        ok = ok && issue(0);
        for (int s = 0; ok && held[s] < nchunk; s ^= 1) {
            ok = issue(s ^ 1) && check(hipEventSynchronize(ev[s]));
            if (!ok) break;
            const size_t off = held[s] * chunk;
            std::memcpy((char*)dst + off, pinned + (2 * (size_t)t + s) * chunk, std::min(chunk, bytes - off));
        }
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
    };
    std::array<std::thread, kThreads> threads;
    for (int t = 1; t < want; ++t) {
        try {
            threads[t] = std::thread(work, t);
        } catch (...) {  // no further thread: those that run take every chunk
            break;
        }
    }
    work(0);
    for (std::thread& t : threads)
        if (t.joinable()) t.join();
    const hipError_t done = hipStreamSynchronize(st);  // an error may have left transfers into the buffers
    (void)hipHostFree(pinned);
    return error != hipSuccess ? (hipError_t)error.load() : done;
}

}  // namespace hfg
