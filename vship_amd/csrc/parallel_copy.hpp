// A fork-join group of worker threads for large memcpy calls (no HIP
// dependency): copy() splits the bytes of one range, or of a list of
// segments, into equal parts cut at 4 KiB boundaries, and the calling thread
// copies the first part itself.
#pragma once
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace vship {

// [begin, end) of part `idx` of `parts` of a `bytes`-long copy; the parts
// cover [0, bytes) without overlap.
inline void copy_part_range(size_t bytes, int idx, int parts, size_t* begin, size_t* end) {
    const size_t per = ((bytes + parts - 1) / parts + 4095) / 4096 * 4096;
    *begin = std::min(bytes, per * idx);
    *end = std::min(bytes, *begin + per);
}

// One contiguous piece of a gathered copy.
struct CopySeg {
    uint8_t* dst;
    const uint8_t* src;
    size_t bytes;
};

// Copies the bytes [b, e) of the concatenation of `segs`.
inline void copy_seg_range(const CopySeg* segs, int n, size_t b, size_t e) {
    size_t s0 = 0;
    for (int i = 0; i < n && s0 < e; i++) {
        const size_t s1 = s0 + segs[i].bytes;
        const size_t lo = std::max(b, s0), hi = std::min(e, s1);
        if (hi > lo) std::memcpy(segs[i].dst + (lo - s0), segs[i].src + (lo - s0), hi - lo);
        s0 = s1;
    }
}

class ParallelCopy {
public:
    explicit ParallelCopy(int threads) : nthreads_(std::max(1, std::min(threads, 64))) {
        for (int i = 1; i < nthreads_; i++) workers_.emplace_back(&ParallelCopy::worker, this, i);
    }
    ~ParallelCopy() {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        go_.notify_all();
        for (auto& t : workers_) t.join();
    }
    ParallelCopy(const ParallelCopy&) = delete;
    ParallelCopy& operator=(const ParallelCopy&) = delete;

    int threads() const { return nthreads_; }

    void copy(void* dst, const void* src, size_t bytes) {
        const CopySeg s{static_cast<uint8_t*>(dst), static_cast<const uint8_t*>(src), bytes};
        copy(&s, 1);
    }

    // Copies every segment; the threads split the segments' total bytes.
    void copy(const CopySeg* segs, int n) {
        size_t total = 0;
        for (int i = 0; i < n; i++) total += segs[i].bytes;
        // below ~1 MiB per extra thread the wake-ups cost more than they save
        if (workers_.empty() || total < ((size_t)1 << 20) * workers_.size()) {
            copy_seg_range(segs, n, 0, total);
            return;
        }
        {
            std::lock_guard<std::mutex> lk(mu_);
            segs_ = segs;
            nseg_ = n;
            total_ = total;
            remaining_ = (int)workers_.size();
            gen_++;
        }
        go_.notify_all();
        part(segs, n, total, 0);
        std::unique_lock<std::mutex> lk(mu_);
        done_.wait(lk, [&] { return remaining_ == 0; });
    }

private:
    void part(const CopySeg* segs, int n, size_t total, int idx) const {
        size_t b, e;
        copy_part_range(total, idx, nthreads_, &b, &e);
        if (e > b) copy_seg_range(segs, n, b, e);
    }

    // Each worker takes every generation: copy() starts the next one only
    // after all workers have finished the last.
    void worker(int idx) {
        uint64_t seen = 0;
        for (;;) {
            const CopySeg* segs;
            int n;
            size_t total;
            {
                std::unique_lock<std::mutex> lk(mu_);
                go_.wait(lk, [&] { return stop_ || gen_ != seen; });
                if (stop_) return;
                seen = gen_;
                segs = segs_;
                n = nseg_;
                total = total_;
            }
            part(segs, n, total, idx);
            {
                std::lock_guard<std::mutex> lk(mu_);
                if (--remaining_ == 0) done_.notify_one();
            }
        }
    }

    const int nthreads_;
    std::vector<std::thread> workers_;
    std::mutex mu_;
    std::condition_variable go_, done_;
    uint64_t gen_ = 0;
    int remaining_ = 0;
    bool stop_ = false;
    const CopySeg* segs_ = nullptr;
    int nseg_ = 0;
    size_t total_ = 0;
};

// Helper threads for one copy at a time that goes chunk by chunk through a
// ring, such as an upload whose chunks cross PCIe while the next ones are
// filled. The callers of all threads may share one team: a copy that finds it
// taken runs on its own thread alone.
class CopyTeam {
public:
    // rows of `bytes` bytes at the two strides (one row: a plain copy)
    struct Piece {
        uint8_t* dst;
        const uint8_t* src;
        size_t bytes;
        int chunk;
        int rows = 1;
        int64_t dst_stride = 0, src_stride = 0;
    };

    // Fewer helpers, or none, where the system gives no more threads.
    explicit CopyTeam(int helpers) {
        threads_.reserve(helpers);
        try {
            for (int i = 0; i < helpers; i++) threads_.emplace_back(&CopyTeam::helper, this);
        } catch (const std::system_error&) {
        }
    }
    ~CopyTeam() {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        go_.notify_all();
        for (auto& t : threads_) t.join();
    }
    CopyTeam(const CopyTeam&) = delete;
    CopyTeam& operator=(const CopyTeam&) = delete;

    // Copies the pieces, which are in order of their chunks 0 .. nchunks - 1,
    // each with at least one piece. On the calling thread, in order:
    // open(c, wait) says whether chunk c may be copied now (wait: blocks until
    // it may), asked only once chunk c - depth is done; done(c) follows its last
    // piece. An exception from either ends the copy and is passed on.
    template <class Open, class Done>
    void run(const std::vector<Piece>& pieces, int nchunks, int depth, Open&& open, Done&& done) {
        Job job(pieces, nchunks);
        std::unique_lock<std::mutex> mine(use_, std::defer_lock);
        if (threads_.empty() || !mine.try_lock()) {
            size_t i = 0;
            for (int c = 0; c < nchunks; c++) {
                open(c, true);
                for (; i < pieces.size() && pieces[i].chunk == c; i++) copy(pieces[i]);
                done(c);
            }
            return;
        }
        post(&job);
        int opened = 0;
        try {
            for (int c = 0; c < nchunks; c++) {
                while (job.left[c].load(std::memory_order_acquire) > 0) {
                    while (opened < std::min(nchunks, c + depth) && open(opened, opened <= c))
                        job.opened.store(++opened, std::memory_order_release);
                    if (!job.take_open(opened)) std::this_thread::yield();
                }
                done(c);
            }
        } catch (...) {
            job.abort.store(true);
            post(nullptr);
            throw;
        }
        post(nullptr);
    }

private:
    struct Job {
        const std::vector<Piece>& pieces;
        std::unique_ptr<std::atomic<int>[]> left;  // pieces of each chunk still to be copied
        std::atomic<int> next{0}, opened{0};
        std::atomic<bool> abort{false};
        Job(const std::vector<Piece>& p, int nchunks) : pieces(p), left(new std::atomic<int>[nchunks]) {
            for (int c = 0; c < nchunks; c++) left[c].store(0, std::memory_order_relaxed);
            for (const Piece& q : p) left[q.chunk].fetch_add(1, std::memory_order_relaxed);
        }
        void finish(int i) {
            copy(pieces[i]);
            left[pieces[i].chunk].fetch_sub(1, std::memory_order_release);
        }
        // the calling thread: one piece, if the next one's chunk is open
        bool take_open(int open) {
            int i = next.load(std::memory_order_relaxed);
            if (i >= (int)pieces.size() || pieces[i].chunk >= open) return false;
            if (next.compare_exchange_strong(i, i + 1)) finish(i);
            return true;
        }
        // a helper: piece after piece, each when its chunk is open
        void help() {
            for (;;) {
                const int i = next.fetch_add(1);
                if (i >= (int)pieces.size()) return;
                while (opened.load(std::memory_order_acquire) <= pieces[i].chunk) {
                    if (abort.load()) return;
                    std::this_thread::yield();
                }
                finish(i);
            }
        }
    };

    static void copy(const Piece& p) {
        for (int r = 0; r < p.rows; r++)
            std::memcpy(p.dst + (int64_t)r * p.dst_stride, p.src + (int64_t)r * p.src_stride, p.bytes);
    }

    // the job helpers may join; nullptr: none, after the last has left
    void post(Job* j) {
        std::unique_lock<std::mutex> lk(mu_);
        job_ = j;
        if (j) {
            gen_++;
            lk.unlock();
            go_.notify_all();
        } else {
            idle_.wait(lk, [&] { return active_ == 0; });
        }
    }

    void helper() {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lk(mu_);
        for (;;) {
            go_.wait(lk, [&] { return stop_ || (job_ && gen_ != seen); });
            if (stop_) return;
            seen = gen_;
            Job* j = job_;
            active_++;
            lk.unlock();
            j->help();
            lk.lock();
            if (--active_ == 0) idle_.notify_all();
        }
    }

    std::vector<std::thread> threads_;
    std::mutex use_;  // held by the copy that has the helpers
    std::mutex mu_;
    std::condition_variable go_, idle_;
    Job* job_ = nullptr;
    uint64_t gen_ = 0;
    int active_ = 0;
    bool stop_ = false;
};

}  // namespace vship
