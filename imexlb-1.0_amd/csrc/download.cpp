// download.cpp -- fields from the device's padded arrays to the caller's dense
// ones.
//
// A single thread that copies whole padded arrays to a vector and picks the
// interior out of it is bound by first touches of that vector and of the
// caller's fresh pages (8193 x 2049: 81 ms for 403 MB).  Here a kernel writes
// runs of interior values straight into pinned buffers, and a few threads, each
// with a buffer of its own, copy them out while the next runs arrive: 11.5 ms
// (35 GB/s); 513 x 129 x 129 49 to 8.4 ms, 401 x 101 0.52 to 0.10 ms.  Small
// fields keep the single copy.
#include "context.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace imexlb {

void Staging::release()
{
    for (int k = 0; k < kWorkers; ++k) {
        if (host[k]) (void)hipHostFree(host[k]);
        if (done[k]) (void)hipEventDestroy(done[k]);
        host[k] = nullptr;
        done[k] = nullptr;
    }
    values = 0;
}

// kWorkers buffers of at least n values; false without memory for them
static bool reserve(Staging &s, int workers, int64_t n)
{
    if (s.values < n) s.release();
    for (int k = 0; k < workers; ++k) {
        if (s.host[k]) continue;
        void *p = nullptr;
        if (hipHostMalloc(&p, size_t(n) * sizeof(double), hipHostMallocDefault) != hipSuccess ||
            hipEventCreateWithFlags(&s.done[k], hipEventDisableTiming) != hipSuccess) {
            if (p) (void)hipHostFree(p);
            s.done[k] = nullptr;
            (void)hipGetLastError();
            s.release();
            return false;
        }
        s.host[k] = static_cast<double *>(p);
        s.values = n;
    }
    return true;
}

bool download_interior(Staging &s, int device, hipStream_t stream, int dim, const KParams &kp,
                       const std::vector<FieldCopy> &fields, hipError_t &err)
{
    // 256 Ki values (2 MiB) a run, and at least two runs of 48 Ki a thread: with
    // fewer values starting a thread costs more than it copies (801 x 201 371
    // us with runs of 8 Ki, 313 with 32, 237 with 64, 299 on one thread; 96
    // arrays of 3 x 118 Ki 37, 33, 37 and 52 ms)
    constexpr int64_t kRun = int64_t(256) << 10, kLeast = int64_t(48) << 10;
    err = hipSuccess;
    const int64_t n = kp.N, total = n * int64_t(fields.size());
    // Few values: the whole padded arrays through a vector cost less than
    // launches and events (us, 61 x 61 34 and 45, 17 x 17 x 17 48 and 59, 151 x
    // 151 62 and 64, 181 x 181 79 and 76), but not copies of up to 16 KiB, which
    // the runtime makes in 23 us each instead of 11 (41 x 41 68 and 44).
    if (kp.plane * int64_t(sizeof(double)) > (int64_t(16) << 10) && total < (int64_t(80) << 10)) return false;
    const int64_t cores = std::max(1u, std::thread::hardware_concurrency());
    const int workers = int(std::clamp<int64_t>(total / (2 * kLeast), 1, std::min<int64_t>(Staging::kWorkers, cores)));
    const int64_t run = std::min(kRun, std::max(kLeast, (total + 2 * workers - 1) / (2 * workers)));
    // (a staging area once made for large runs serves small ones too)
    if (!reserve(s, workers, std::max(run, s.values))) return false;
    const int64_t per = (n + run - 1) / run, runs = per * int64_t(fields.size());
    std::atomic<int64_t> next{0};
    std::vector<hipError_t> bad(size_t(workers), hipSuccess);
    const auto work = [&](int w) noexcept {
        hipError_t e = hipSetDevice(device);
        for (int64_t r; e == hipSuccess && (r = next.fetch_add(1)) < runs;) {
            const FieldCopy &f = fields[size_t(r / per)];
            const int64_t first = r % per * run, count = std::min(run, n - first);
            e = launch_pack(dim, kp, f.from, first, count, s.host[w], stream);
            if (e == hipSuccess) e = hipEventRecord(s.done[w], stream);
            if (e == hipSuccess) e = hipEventSynchronize(s.done[w]);
            if (e == hipSuccess) std::memcpy(f.to + first, s.host[w], size_t(count) * sizeof(double));
        }
        bad[size_t(w)] = e;
    };
    std::vector<std::thread> threads;
    threads.reserve(size_t(workers));
    for (int w = 1; w < workers; ++w) {
        try {
            threads.emplace_back(work, w);
        } catch (...) {  // no more threads: those that run take all the runs
            break;
        }
    }
    work(0);
    for (std::thread &t : threads) t.join();
    for (hipError_t e : bad)
        if (e != hipSuccess) err = e;
    return true;
}

}  // namespace imexlb
