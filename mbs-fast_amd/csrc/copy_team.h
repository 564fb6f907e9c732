// copy_team.h -- host threads that share a context's large copies.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace mbs {

// Host threads of a context for its large copies: three beside the caller, started
// with the first such copy and joined with the context.
class CopyTeam {
public:
    enum { kHelpers = 3, kLeast = 1 << 19 };  // 512 KiB: 50 us alone, 30 shared
    explicit CopyTeam(int helpers = kHelpers) : helpers_(helpers) {}
    // The bytes of one of `parts` equal parts, a whole number of pages: together they
    // hold every byte (the last ones may be short or empty).
    static size_t share(size_t bytes, int parts)
    {
        return ((bytes + parts - 1) / parts + 4095) / 4096 * 4096;
    }
    ~CopyTeam()
    {
        {
            std::lock_guard<std::mutex> lock(m_);
            stop_ = true;
        }
        wake_.notify_all();
        for (std::thread &t : threads_)
            t.join();
    }
    // Copies bytes (or adds FP64 values), in equal parts; alone if no thread can be
    // started.
    void copy(void *dst, const void *src, size_t bytes, bool add = false)
    {
        if (bytes < kLeast) {
            run(0, (unsigned char *)dst, (const unsigned char *)src, bytes, bytes, add);
            return;
        }
        if (threads_.empty() && !alone_) {
            try {
                threads_.reserve(helpers_);
                for (int i = 0; i < helpers_; ++i)
                    threads_.emplace_back([this, i] { serve(i); });
            } catch (...) {
                alone_ = threads_.empty();
            }
        }
        const int parts = (int)threads_.size() + 1;
        const size_t part = share(bytes, parts);
        {
            std::lock_guard<std::mutex> lock(m_);
            dst_ = (unsigned char *)dst;
            src_ = (const unsigned char *)src;
            bytes_ = bytes;
            part_ = part;
            add_ = add;
            left_ = parts - 1;
            ++round_;
        }
        wake_.notify_all();
        run(parts - 1, dst_, src_, bytes, part, add);
        std::unique_lock<std::mutex> lock(m_);
        done_.wait(lock, [this] { return left_ == 0; });
    }

private:
    static void run(int i, unsigned char *dst, const unsigned char *src, size_t bytes, size_t part,
                    bool add)
    {
        const size_t lo = std::min(bytes, part * i), hi = std::min(bytes, lo + part);
        if (lo >= hi)
            return;
        if (!add) {
            std::memcpy(dst + lo, src + lo, hi - lo);
            return;
        }
        double *d = (double *)(dst + lo);
        const double *s = (const double *)(src + lo);
        for (size_t n = (hi - lo) / sizeof(double), e = 0; e < n; ++e)
            d[e] += s[e];
    }
    void serve(int i)
    {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lock(m_);
        for (;;) {
            wake_.wait(lock, [&] { return stop_ || round_ != seen; });
            if (stop_)
                return;
            seen = round_;
            unsigned char *dst = dst_;
            const unsigned char *src = src_;
            const size_t bytes = bytes_, part = part_;
            const bool add = add_;
            lock.unlock();
            run(i, dst, src, bytes, part, add);
            lock.lock();
            if (--left_ == 0)
                done_.notify_one();
        }
    }
    const int helpers_;
    std::vector<std::thread> threads_;
    std::mutex m_;
    std::condition_variable wake_, done_;
    bool stop_ = false, alone_ = false, add_ = false;
    uint64_t round_ = 0;
    int left_ = 0;
    unsigned char *dst_ = nullptr;
    const unsigned char *src_ = nullptr;
    size_t bytes_ = 0, part_ = 0;
};

}  // namespace mbs
