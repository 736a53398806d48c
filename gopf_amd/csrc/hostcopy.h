// hostcopy.h -- moving whole fields between a caller's pageable arrays and the device.
//
// A pageable hipMemcpy of a field goes through the runtime's own staging on one thread, the
// conversion to or from the caller's complex128 is another pass over a temporary, and a fresh
// array's page faults are taken one by one (256^3 FP32 read back in about 22 ms, now 4.4;
// the wire needs 1.3).  HostStage copies the chunks of a large field into pinned memory while a few
// threads convert the chunks that have arrived.  The pinned memory belongs to the object (at most kWorkers kSlots
// chunks) and is freed with it; one call at a time per object, as for every handle.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <exception>
#include <mutex>
#include <system_error>
#include <thread>
#include <type_traits>
#include <vector>

#include "common.h"

namespace gpf {

class HostStage {
    struct Nothing {
        void operator()() const {}
    };

public:
    HostStage() = default;
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    ~HostStage() { release(); }

    // use(src, off, len) for every chunk of the bytes at dev, off and len multiples of 16 but at the
    // end, from several threads at once; returns when all are used.  ready() runs before the first
    // use, once the stream's work has ended: for one copy with it (a wait of its own cost 7 us of a
    // 32^2 read-back), for chunks before the first of them, so that it may throw or wait itself
    template <typename F, typename R>
    void download(const void* dev, size_t bytes, hipStream_t st, F&& use, R&& ready) {
        if (bytes <= kDirect) {
            if (small_.size() < bytes) wait_small(st), small_.resize(bytes);
            small_busy_ = true;
            HIPCHK(hipMemcpyAsync(small_.data(), dev, bytes, hipMemcpyDeviceToHost, st));
            wait_small(st);
            ready();
            use(static_cast<const char*>(small_.data()), (size_t)0, bytes);
            return;
        }
        if constexpr (!std::is_same<std::decay_t<R>, Nothing>::value) {
            HIPCHK(hipStreamSynchronize(st));
            ready();
        }
        const Plan p = plan(bytes);
        auto issue = [&](size_t c) {
            const size_t off = c * p.chunk, len = std::min(p.chunk, bytes - off);
            HIPCHK(hipMemcpyAsync(slot(p, c), static_cast<const char*>(dev) + off, len, hipMemcpyDeviceToHost, st));
            HIPCHK(hipEventRecord(ev_[p.index(c)], st));
            used_[p.index(c)] = 1;  // should the call end before its use
        };
        for (size_t c = 0; c < std::min(p.chunks, (size_t)p.slots); ++c) issue(c);
        run(p, st, [&](size_t c) {
            HIPCHK(hipEventSynchronize(ev_[p.index(c)]));
            const size_t off = c * p.chunk;
            use(static_cast<const char*>(slot(p, c)), off, std::min(p.chunk, bytes - off));
            if (c + p.slots < p.chunks) issue(c + p.slots);
        });
    }

    template <typename F>
    void download(const void* dev, size_t bytes, hipStream_t st, F&& use) {
        download(dev, bytes, st, use, Nothing{});
    }

    // fill(dst, off, len) for every chunk, copied to dev in stream order; returns when every chunk is
    // filled and on its way (the copies end in stream order)
    template <typename F>
    void upload(void* dev, size_t bytes, hipStream_t st, F&& fill) {
        if (bytes <= kDirect) {
            wait_small(st);
            if (small_.size() < bytes) small_.resize(bytes);
            fill(small_.data(), (size_t)0, bytes);
            small_busy_ = true;
            HIPCHK(hipMemcpyAsync(dev, small_.data(), bytes, hipMemcpyHostToDevice, st));
            return;
        }
        const Plan p = plan(bytes);
        run(p, st, [&](size_t c) {
            const size_t off = c * p.chunk, len = std::min(p.chunk, bytes - off);
            // a slot is free once the copy before it has ended
            if (used_[p.index(c)]) HIPCHK(hipEventSynchronize(ev_[p.index(c)]));
            fill(static_cast<char*>(slot(p, c)), off, len);
            HIPCHK(hipMemcpyAsync(static_cast<char*>(dev) + off, slot(p, c), len, hipMemcpyHostToDevice, st));
            HIPCHK(hipEventRecord(ev_[p.index(c)], st));
            used_[p.index(c)] = 1;
        });
    }

private:
    // Starting a thread costs 20 to 50 us, and about 250 more where the host did something else
    // between the calls: one thread per MB, and up to kDirect one pageable copy, from where the
    // slower of these starts still costs less (us with one copy; a thread per MB, and the same after
    // a pause; eight threads from 256 KB on, after pauses 50 to 150 more: complex128 transform in FP32
    // of 512^2, 2 MB, 369; 257 and 503; 421; FP64 of 512^2, 4 MB, 594; 475 and 554; 705).  FP32 field
    // of 1024^2, 4 MB, into a mapped array and a fresh one: 582 and 1550; 464 and 761; 834 and 808.
    // Threads kept waiting between the calls took longer to wake than new ones to start (192^2
    // transform 496 us, one copy 96).
    // Chunks of 1 MB against 512 KB: 128^3 complex128 transform 2.4 against 3.2 ms, 256^3 FP32 field
    // 4.4 against 4.8 ms (eight threads; 5.8 ms with four, 4.0 with twelve).
    static constexpr size_t kDirect = (size_t)3584 << 10, kChunkMax = (size_t)1 << 20;
    static constexpr int kWorkers = 8, kSlots = 2;
    struct Plan {
        size_t chunk = 0, chunks = 0;
        int workers = 1, slots = 1;
        int index(size_t c) const { return (int)(c % slots); }
    };

    void wait_small(hipStream_t st) {
        if (small_busy_) HIPCHK(hipStreamSynchronize(st));
        small_busy_ = false;
    }

    // chunk c belongs to worker c mod workers and slot c mod slots (slots a multiple of workers or
    // one per chunk), so a slot is only ever used by one worker
    Plan plan(size_t bytes) {
        Plan p;
        const int cores = std::max(1, (int)std::thread::hardware_concurrency());
        p.workers = (int)std::clamp<size_t>(bytes >> 20, 2, std::min(kWorkers, std::max(cores, 2)));
        p.chunk = (std::min(bytes / (p.workers * kSlots), kChunkMax) + 4095) / 4096 * 4096;
        p.chunks = (bytes + p.chunk - 1) / p.chunk;
        p.slots = (int)std::min<size_t>((size_t)p.workers * kSlots, p.chunks);
        if (p.slots % p.workers) p.slots = p.workers;
        const size_t want = p.chunk * p.slots;
        if (cap_ < want) {
            release();
            HIPCHK(hipHostMalloc(reinterpret_cast<void**>(&buf_), want, hipHostMallocDefault));
            cap_ = want;
        }
        if (p.chunk != last_chunk_ || p.slots != last_slots_) {
            // other slots than the last call's: its uploads still read them
            for (size_t i = 0; i < ev_.size(); ++i)
                if (used_[i]) HIPCHK(hipEventSynchronize(ev_[i]));
            last_chunk_ = p.chunk;
            last_slots_ = p.slots;
        }
        while ((int)ev_.size() < p.slots) {
            hipEvent_t e;
            HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            used_.push_back(0);
            ev_.push_back(e);
        }
        return p;
    }
    void* slot(const Plan& p, size_t c) const { return buf_ + (size_t)p.index(c) * p.chunk; }

    template <typename F>
    void run(const Plan& p, hipStream_t st, F&& work) {
        std::exception_ptr err;
        std::mutex mu;
        auto loop = [&](int w) {
            try {
                for (size_t c = w; c < p.chunks; c += p.workers) work(c);
            } catch (...) {
                std::lock_guard<std::mutex> g(mu);
                if (!err) err = std::current_exception();
            }
        };
        int dev = 0;
        if (p.workers > 1) HIPCHK(hipGetDevice(&dev));
        std::vector<std::thread> th;
        int w = 1;
        try {
            for (; w < p.workers; ++w)
                th.emplace_back([&, w] {
                    if (hipSetDevice(dev) == hipSuccess) {
                        loop(w);
                    } else {
                        std::lock_guard<std::mutex> g(mu);
                        if (!err) err = std::make_exception_ptr(Error(GPF_EDEVICE, "hipSetDevice failed"));
                    }
                });
        } catch (const std::system_error&) {
            // no more threads: the caller takes the chunks left
        }
        loop(0);
        for (; w < p.workers; ++w) loop(w);
        for (auto& t : th) t.join();
        if (err) {
            (void)hipStreamSynchronize(st);  // no copy may outlive the buffers it names
            std::rethrow_exception(err);
        }
    }

    void release() {
        for (auto e : ev_) (void)hipEventDestroy(e);
        ev_.clear();
        used_.clear();
        if (buf_) (void)hipHostFree(buf_);  // waits for the device
        buf_ = nullptr;
        cap_ = 0;
    }

    std::vector<char> small_;  // the host's side of one pageable copy
    bool small_busy_ = false;  // a copy may still read or write it
    char* buf_ = nullptr;
    size_t cap_ = 0;
    std::vector<hipEvent_t> ev_;
    size_t last_chunk_ = 0;
    int last_slots_ = 0;
    std::vector<char> used_;  // the slot's event has been recorded
};

}  // namespace gpf
