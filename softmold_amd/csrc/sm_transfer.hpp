// Device-to-host results of a context: a kernel packs what the caller asked for straight into
// pinned host memory, and the host unpacks it into the caller's buffers.
//
// What bounds it: a small result costs its round trips, a large one the caller's fresh pages.
// One pack kernel and one event take 13 us on an MI355X where every pageable copy takes 25 us
// (a download was five of them); at 3M beads the 144 MB cross the bus in 3 ms, but one thread
// fills the 216 MB of doubles in 46 ms, eight in 10 ms.  Large states therefore go in chunks
// through pinned buffers while up to kWorkers threads unpack the chunk before.
#pragma once
#include "sm_errors.hpp"
#include "sm_internal.hpp"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace smdev {

class HostLink {
public:
    // Chunks: beads that a pinned buffer holds, and buffers.  A context's first transfer allocates
    // them: 45 us for 1.5 MiB, 290 and more from 3 MiB on, which made the first download of 72k
    // beads 950 us where pageable copies took 600 (335 with the short ones).  A large download
    // pays little for that and more for each chunk that is handed over: 240k beads 1050 to 1100
    // us long, 1050 to 1500 short; 1M beads 3.0 and 4.1 ms.
    struct Chunks {
        int beads, buffers, count;
        explicit Chunks(int n)
            : beads(n > 196608 ? 65536 : 32768), buffers(n > 196608 ? 2 : 4), count((n + beads - 1) / beads)
        {
        }
    };
    static constexpr int kBuffers = 4;            // at most
    static constexpr int kThreadBeads = 65536;    // fewer beads are unpacked by the caller alone
    static constexpr int kWorkers = 8;
    static constexpr size_t kResults = 4;         // doubles a replica that one fetch returns, at most

    // With the context's device current: what every call needs -- the events, which belong to the
    // device that is current when they are made, and the buffer of the largest result of
    // `replicas` replicas -- so that no call depends on the device current then, and a result's
    // first fetch allocates nothing.
    void create(int replicas)
    {
        check(hipGetDevice(&device_), "device");
        for (hipEvent_t &e : ev_) check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "event");
        room_ = kResults * (size_t)replicas;
        check(hipHostMalloc(reinterpret_cast<void **>(&head_), (room_ + 1) * sizeof(double), hipHostMallocDefault), "buffer");
    }

    void destroy()
    {
        for (void *&p : buf_) {
            if (p) (void)hipHostFree(p);
            p = nullptr;
        }
        for (hipEvent_t &e : ev_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (head_) (void)hipHostFree(head_);
        head_ = nullptr;
    }

    // `count` doubles from device memory with the context's state flags: returns the flags
    int fetch(hipStream_t st, const DevGlobal *glob, const double *src, size_t count, double *dst)
    {
        if (count > room_) throw smapi::ApiError(SM_ERR_STATE, "a result larger than its buffer");
        launch_post(st, src, count, glob, head_);
        check(hipGetLastError(), "post");
        finish(st, 0);
        if (count) std::memcpy(dst, head_ + 1, count * sizeof(double));
        return flags();
    }

    // The box lengths of every replica and the state flags.
    int fetch_boxes(hipStream_t st, const DevGlobal *glob, const DevRep *reps, int nrep, double *box)
    {
        launch_pack(st, 0, 0, PackSrc{nullptr, nullptr, nullptr}, nullptr, reps, nrep, glob, head_);
        check(hipGetLastError(), "pack");
        finish(st, 0);
        std::memcpy(box, head_ + 1, 3 * sizeof(double) * (size_t)nrep);
        return flags();
    }

    // n beads' positions and up to two float4 arrays as n x 3 doubles (a NULL destination
    // skips its source), the boxes if box, and the state flags.
    int fetch_beads(hipStream_t st, int n, const PackSrc &src, double *pos, double *a, double *b,
                    const DevGlobal *glob, const DevRep *reps, int nrep, double *box)
    {
        const PackSrc s{pos ? src.beads : nullptr, a ? src.a : nullptr, b ? src.b : nullptr};
        const Chunks ch(n);
        const int chunks = ch.count;
        buffers(std::min(n, ch.beads), std::min(chunks, ch.buffers));
        auto launch = [&](int c) {
            const int first = c * ch.beads, count = std::min(ch.beads, n - first);
            launch_pack(st, first, count, s, static_cast<double *>(buf_[c % ch.buffers]), reps, c == 0 ? nrep : 0, glob,
                        c == 0 ? head_ : nullptr);
            check(hipGetLastError(), "pack");
            check(hipEventRecord(ev_[c % ch.buffers], st), "event");
        };
        auto wait = [&](int c) { check(hipEventSynchronize(ev_[c % ch.buffers]), "event"); };
        // beads [count i / parts, count (i + 1) / parts) of chunk c into the caller's arrays
        auto unpack = [&](int c, int i, int parts) {
            const int first = c * ch.beads, count = std::min(ch.beads, n - first);
            const size_t e0 = 3 * ((size_t)count * i / parts), e1 = 3 * ((size_t)count * (i + 1) / parts);
            const double *p = static_cast<const double *>(buf_[c % ch.buffers]);
            const float *f = reinterpret_cast<const float *>(p + (s.beads ? 3 * (size_t)count : 0));
            const size_t o = 3 * (size_t)first;
            if (s.beads) std::memcpy(pos + o + e0, p + e0, (e1 - e0) * sizeof(double));
            if (s.a)
                for (size_t e = e0; e < e1; e++) a[o + e] = f[e];
            if (s.a) f += 3 * (size_t)count;
            if (s.b)
                for (size_t e = e0; e < e1; e++) b[o + e] = f[e];
        };
        const int want = n < kThreadBeads ? 1 : std::max(1, std::min(kWorkers, (int)std::thread::hardware_concurrency() / 2));
        std::atomic<int> ready{0}, done{0};
        // The workers sleep until the first chunk is there: the GPU may have any amount of queued
        // work before it (seven of them polling took as many cores for a whole stretch of steps).
        // After it, chunks come as fast as they are unpacked, and they poll.
        std::mutex mu;
        std::condition_variable wake;
        int size = 0;   // parts, once the first chunk is there
        std::atomic<bool> quit{false};
        const auto work = [&](int i) {
            int parts;
            {
                std::unique_lock<std::mutex> lock(mu);
                wake.wait(lock, [&] { return size != 0 || quit.load(); });
                parts = size;
            }
            for (int c = 0; c < chunks; c++) {
                while (ready.load(std::memory_order_acquire) <= c)
                    if (quit.load()) return;
                    else std::this_thread::yield();
                unpack(c, i, parts);
                done.fetch_add(1, std::memory_order_release);
            }
        };
        std::vector<std::thread> team;
        struct Join {   // the last of what the workers use, so the first to go
            std::vector<std::thread> &t;
            std::mutex &mu;
            std::condition_variable &wake;
            std::atomic<bool> &quit;
            ~Join()
            {
                {
                    std::lock_guard<std::mutex> lock(mu);
                    quit.store(true);
                }
                wake.notify_all();
                for (auto &x : t) x.join();
            }
        };
        {
            Join join{team, mu, wake, quit};
            launch(0);
            try {
                team.reserve(want);
                for (int i = 1; i < want; i++) team.emplace_back(work, i);
            } catch (const std::exception &) {   // no thread, or no memory for one: those there are
            }
            const int parts = 1 + (int)team.size();
            for (int c = 1; c < std::min(chunks, ch.buffers); c++) launch(c);
            wait(0);
            {
                std::lock_guard<std::mutex> lock(mu);
                size = parts;
            }
            wake.notify_all();
            for (int c = 0; c < chunks; c++) {
                if (c > 0) wait(c);
                ready.store(c + 1, std::memory_order_release);
                unpack(c, 0, parts);
                while (done.load(std::memory_order_acquire) < (c + 1) * (parts - 1)) std::this_thread::yield();
                if (c + ch.buffers < chunks) launch(c + ch.buffers);
            }
        }
        if (box) std::memcpy(box, head_ + 1, 3 * sizeof(double) * (size_t)nrep);
        return flags();
    }

    // the count of fallbacks (DevGlobal) that came with the last result
    uint32_t fallbacks() const { return (uint32_t)((unsigned long long)word() >> 32); }

    // reps[r].scale = scale[3r ..]; the caller's array is free again on return, the buffer after
    // the next fetch
    void send_scale(hipStream_t st, DevRep *reps, int nrep, const double *scale)
    {
        std::memcpy(head_ + 1, scale, 3 * sizeof(double) * (size_t)nrep);
        launch_set_scale(st, reps, nrep, head_ + 1);
        check(hipGetLastError(), "scale");
    }

    // beads[i].x, y, z = pos[3 i ..] for n beads; the caller's array is free again on return
    void send_positions(hipStream_t st, int n, const double *pos, Bead *beads)
    {
        const Chunks ch(n);
        const int chunks = ch.count;
        buffers(std::min(n, ch.beads), std::min(chunks, ch.buffers));
        for (int c = 0; c < chunks; c++) {
            const int first = c * ch.beads, count = std::min(ch.beads, n - first);
            check(hipEventSynchronize(ev_[c % ch.buffers]), "event");   // the buffer's last kernel is done
            std::memcpy(buf_[c % ch.buffers], pos + 3 * (size_t)first, 3 * sizeof(double) * (size_t)count);
            launch_set_positions(st, first, count, static_cast<const double *>(buf_[c % ch.buffers]), beads);
            check(hipGetLastError(), "unpack");
            check(hipEventRecord(ev_[c % ch.buffers], st), "event");
        }
    }

private:
    void *buf_[kBuffers] = {};
    size_t beads_[kBuffers] = {};
    double *head_ = nullptr;      // flags and fallbacks, then room_ doubles
    size_t room_ = 0;
    int device_ = 0;              // the context's
    hipEvent_t ev_[kBuffers] = {};

    static void check(hipError_t e, const char *what)
    {
        if (e != hipSuccess)
            throw smapi::ApiError(SM_ERR_HIP, std::string(hipGetErrorName(e)) + " in a " + what + " of a result transfer");
    }
    void buffers(int beads, int want)
    {
        for (int i = 0; i < want; i++) {
            if (buf_[i] && (size_t)beads <= beads_[i]) continue;
            OnDevice here(device_);
            if (buf_[i]) (void)hipHostFree(buf_[i]);
            buf_[i] = nullptr;
            beads_[i] = 0;
            check(hipHostMalloc(&buf_[i], (size_t)std::max(beads, 1) * kPackBytes, hipHostMallocDefault), "buffer");
            beads_[i] = (size_t)beads;
        }
    }
    // the context's device current, then again the caller's
    struct OnDevice {
        int was = -1;
        explicit OnDevice(int device)
        {
            int now;
            check(hipGetDevice(&now), "device");
            if (now == device) return;
            check(hipSetDevice(device), "device");
            was = now;
        }
        ~OnDevice()
        {
            if (was >= 0) (void)hipSetDevice(was);
        }
    };
    void finish(hipStream_t st, int e)
    {
        check(hipEventRecord(ev_[e], st), "event");
        check(hipEventSynchronize(ev_[e]), "event");
    }
    long long word() const
    {
        long long f;
        std::memcpy(&f, head_, sizeof f);
        return f;
    }
    int flags() const { return (int)word(); }
};

}  // namespace smdev
