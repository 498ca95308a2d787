// mm_readback.h -- large states from the device to the caller's doubles.
// Included after mm_conv.h (MM_HIP).
#ifndef MM_READBACK_H
#define MM_READBACK_H

#include <algorithm>
#include <condition_variable>
#include <cstddef>
#include <map>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include <hip/hip_runtime.h>

// Large device arrays to host doubles: pieces go through a few pinned buffers
// in the state's own precision, and host threads widen (or copy) each piece
// into the caller's array while the next ones are on their way.  A pageable
// copy of doubles is staged by the runtime on one thread; that took 18.8 ms
// for 512x512x32 (FP32 and FP64), 5.0 for 1024x1024x2 and 1.4 for 256x256x16,
// this takes 4.9 / 7.4, 1.5 / 2.2 and 0.5 / 0.85 ms.  One set of buffers per
// device serves all steppers that read large states, one read at a time, and
// goes with the last of them.
struct Readback {
    // of doubles: 200x200x8 (7.7 MB) reads in 0.47 ms either way, 256x256x6
    // (9.4 MB) in 0.27 / 0.45 ms instead of 0.55
    static constexpr size_t MIN_BYTES = (size_t)8 << 20;
    static constexpr size_t PIECE_BYTES = (size_t)2 << 20;
    static constexpr int NBUF = 4, NTHR = 8;
    void *buf[NBUF] = {};
    hipEvent_t ev[NBUF] = {};
    std::mutex busy;

    // the current device's buffers
    static std::shared_ptr<Readback> get()
    {
        static std::mutex mu;
        static std::map<int, std::weak_ptr<Readback>> all;
        int dev = 0;
        MM_HIP(hipGetDevice(&dev));
        std::lock_guard<std::mutex> lk(mu);
        std::shared_ptr<Readback> r = all[dev].lock();
        if (!r) {
            r = std::make_shared<Readback>();
            all[dev] = r;
        }
        return r;
    }

    Readback()
    {
        try {
            for (int b = 0; b < NBUF; ++b) {
                MM_HIP(hipHostMalloc(&buf[b], PIECE_BYTES, hipHostMallocDefault));
                MM_HIP(hipEventCreateWithFlags(&ev[b], hipEventDisableTiming));
            }
        } catch (...) {
            release();
            throw;
        }
    }
    ~Readback() { release(); }
    Readback(const Readback &) = delete;
    void release()
    {
        for (int b = 0; b < NBUF; ++b) {
            if (ev[b]) (void)hipEventDestroy(ev[b]);
            if (buf[b]) (void)hipHostFree(buf[b]);
            ev[b] = nullptr;
            buf[b] = nullptr;
        }
    }

    // false: the host gave no thread, nothing was read
    template <typename T> bool run(double *dst, const T *src, size_t cnt, hipStream_t s)
    {
        constexpr size_t PIECE = PIECE_BYTES / sizeof(T);
        std::lock_guard<std::mutex> one(busy);
        const size_t np = (cnt + PIECE - 1) / PIECE;
        std::mutex mu;
        std::condition_variable cv;
        size_t landed = 0;          // pieces in their buffers
        bool quit = false;
        int nthr = 0;               // set before the first piece lands
        std::vector<int> done(np, 0);  // threads finished with a piece
        std::vector<std::thread> thr;
        auto work = [&](int t) {
            for (size_t i = 0; i < np; ++i) {
                {
                    std::unique_lock<std::mutex> lk(mu);
                    cv.wait(lk, [&] { return quit || landed > i; });
                    if (landed <= i) return;
                }
                const size_t n = std::min(PIECE, cnt - i * PIECE);
                const size_t a = n * t / nthr, e = n * (t + 1) / nthr;
                const T *in = (const T *)buf[i % NBUF];
                double *out = dst + i * PIECE;
                for (size_t j = a; j < e; ++j) out[j] = (double)in[j];
                {
                    std::lock_guard<std::mutex> lk(mu);
                    if (++done[i] == nthr) cv.notify_all();
                }
            }
        };
        // every exit ends and joins the threads, and no copy into the buffers
        // is left in flight
        struct Join {
            std::mutex &mu;
            std::condition_variable &cv;
            bool &quit;
            std::vector<std::thread> &thr;
            hipStream_t s;
            ~Join()
            {
                {
                    std::lock_guard<std::mutex> lk(mu);
                    quit = true;
                }
                cv.notify_all();
                for (std::thread &t : thr) t.join();
                (void)hipStreamSynchronize(s);
            }
        } join{mu, cv, quit, thr, s};
        thr.reserve(NTHR);
        try {
            for (int t = 0; t < NTHR; ++t) thr.emplace_back(work, t);
        } catch (const std::system_error &) {
            if (thr.empty()) return false;  // with fewer threads it goes on
        }
        nthr = (int)thr.size();
        auto issue = [&](size_t i) {
            const size_t n = std::min(PIECE, cnt - i * PIECE);
            MM_HIP(hipMemcpyAsync(buf[i % NBUF], src + i * PIECE, n * sizeof(T), hipMemcpyDeviceToHost, s));
            MM_HIP(hipEventRecord(ev[i % NBUF], s));
        };
        for (size_t i = 0; i < std::min<size_t>(np, NBUF); ++i) issue(i);
        for (size_t i = 0; i < np; ++i) {
            MM_HIP(hipEventSynchronize(ev[i % NBUF]));
            {
                std::lock_guard<std::mutex> lk(mu);
                landed = i + 1;
            }
            cv.notify_all();
            // the buffer of piece i + NBUF - 1 is piece i - 1's: refill it
            // once that is through
            if (i >= 1 && i - 1 + NBUF < np) {
                std::unique_lock<std::mutex> lk(mu);
                cv.wait(lk, [&] { return done[i - 1] == nthr; });
                lk.unlock();
                issue(i - 1 + NBUF);
            }
        }
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&] { return done[np - 1] == nthr; });
        return true;
    }
};

// One owner's access to the pieces.  read() is false if they cannot be had (no
// pinned memory, no events on the stream's device, no thread); the caller then
// copies its own way.  What failed once is not tried again.
class StateReader {
    std::mutex mu;
    std::shared_ptr<Readback> rb;
    bool off = false;

  public:
    template <typename T> bool read(double *dst, const T *src, size_t cnt, hipStream_t s)
    {
        std::shared_ptr<Readback> r;
        try {
            {
                std::lock_guard<std::mutex> lk(mu);
                if (off) return false;
                if (!rb) rb = Readback::get();
                r = rb;
            }
            if (r->run(dst, src, cnt, s)) return true;
        } catch (const std::exception &) {
            (void)hipGetLastError();
        }
        std::lock_guard<std::mutex> lk(mu);
        off = true;
        rb.reset();
        return false;
    }
};

#endif
