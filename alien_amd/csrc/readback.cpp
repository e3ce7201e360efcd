// readback.cpp — pinned transfer buffers and the chunked read-back of records.
#include "readback.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "worldset.hpp"

namespace alien {

namespace {
struct Pool {
    std::mutex mutex;
    std::vector<void*> kept;
};
// (never destroyed: buffers still kept at the end go with the process)
Pool& pool() {
    static Pool* p = new Pool;
    return *p;
}
}  // namespace

PinnedBuffer::PinnedBuffer() {
    {
        std::lock_guard<std::mutex> lock(pool().mutex);
        if (!pool().kept.empty()) {
            p_ = pool().kept.back();
            pool().kept.pop_back();
        }
    }
    // (portable: the pool serves every device of the process)
    if (!p_) check_hip(hipHostMalloc(&p_, kBytes, hipHostMallocPortable), "hipHostMalloc");
}

PinnedBuffer::~PinnedBuffer() {
    {
        std::lock_guard<std::mutex> lock(pool().mutex);
        if (pool().kept.size() < kKept) {
            pool().kept.push_back(p_);
            return;
        }
    }
    (void)hipHostFree(p_);
}

// A chunk goes kernel -> pinned buffer -> caller's memory.  Its second half is the slow one: pages the
// caller has not touched yet are faulted in at about 5 GB/s by one thread (4 KiB pages), 22 GB/s by
// six, while the link delivers 55 GB/s; so chunks are handed to up to six workers, each with a buffer
// of its own, and one worker's copy hides the others' kernels.  One worker per 2 MiB: starting a
// thread costs about 20 us, the time in which one copies 0.1 to 0.5 MB.
void read_records(size_t n, size_t size, void* out, hipStream_t s,
                  const std::function<void(size_t, size_t, void*)>& pack) {
    if (n == 0) return;
    // (whole workgroups of records per chunk)
    const size_t most = std::max<size_t>(256, PinnedBuffer::kBytes / size / 256 * 256);
    const size_t cores = std::max<size_t>(1, std::thread::hardware_concurrency());
    const size_t workers = std::max<size_t>(1, std::min({size_t(6), cores, n * size / PinnedBuffer::kBytes}));
    const size_t chunks = (n + most - 1) / most;
    std::atomic<size_t> next{0};
    std::atomic<bool> failed{false};
    std::exception_ptr error;
    std::mutex errorMutex;
    int device = 0;
    check_hip(hipGetDevice(&device), "hipGetDevice");
    auto work = [&](bool own) {
        try {
            if (own) check_hip(hipSetDevice(device), "hipSetDevice");
            PinnedBuffer buffer;
            hipEvent_t done = nullptr;
            if (chunks > 1) check_hip(hipEventCreateWithFlags(&done, hipEventDisableTiming), "hipEventCreate");
            // (after a failure nothing writes to the buffer any more when it goes back to the pool)
            struct Guard {
                hipEvent_t& done;
                hipStream_t s;
                bool inFlight;
                ~Guard() {
                    if (inFlight) (void)hipStreamSynchronize(s);
                    if (done) (void)hipEventDestroy(done);
                }
            } guard{done, s, false};
            for (size_t c = next++; c < chunks && !failed; c = next++) {
                const size_t first = c * most, count = std::min(most, n - first);
                guard.inFlight = true;
                pack(first, count, buffer.data());
                check_hip(hipGetLastError(), "pack kernel");
                if (done) {
                    check_hip(hipEventRecord(done, s), "hipEventRecord");
                    check_hip(hipEventSynchronize(done), "hipEventSynchronize");
                } else {
                    check_hip(hipStreamSynchronize(s), "hipStreamSynchronize");
                }
                guard.inFlight = false;
                std::memcpy(static_cast<char*>(out) + first * size, buffer.data(), count * size);
            }
        } catch (...) {
            failed = true;
            std::lock_guard<std::mutex> lock(errorMutex);
            if (!error) error = std::current_exception();
        }
    };
    std::vector<std::thread> others;
    others.reserve(workers);
    for (size_t t = 1; t < workers; ++t) {
        try {
            others.emplace_back(work, true);
        } catch (...) {
            break;  // no more threads, or no memory for one: the ones there are do the rest
        }
    }
    work(false);
    for (auto& t : others) t.join();
    if (error) std::rethrow_exception(error);
}

// One thread per 16384 entries: the work on an entry is 5 to 60 ns, and starting and joining one takes 50 to 200 us
// where the process holds a device (20,971 cells on one thread 0.39 ms, on two 0.4 to 0.9; 65,536 on four 1.5, 209,606
// in bodies on eight 2.5 instead of 12).
void for_ranges(size_t n, const std::function<void(size_t, size_t)>& f) {
    const size_t cores = std::max<size_t>(1, std::thread::hardware_concurrency());
    const size_t pieces = std::max<size_t>(1, std::min({size_t(8), cores, n / 16384}));
    if (pieces == 1) return f(0, n);
    std::vector<std::exception_ptr> errors(pieces);
    auto work = [&](size_t k) {
        try {
            f(n * k / pieces, n * (k + 1) / pieces);
        } catch (...) {
            errors[k] = std::current_exception();
        }
    };
    std::vector<std::thread> others;
    others.reserve(pieces);
    size_t started = 1;
    for (; started < pieces; ++started) {
        try {
            others.emplace_back(work, started);
        } catch (...) {
            break;  // no more threads, or no memory for one: the pieces left are done here
        }
    }
    work(0);
    for (size_t k = started; k < pieces; ++k) work(k);
    for (auto& t : others) t.join();
    for (const auto& e : errors)
        if (e) std::rethrow_exception(e);
}

}  // namespace alien
