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

    // Whether a copy has the helpers at this moment.
    bool taken() {
        if (threads_.empty()) return false;
        const std::unique_lock<std::mutex> lk(use_, std::try_to_lock);
        return !lk.owns_lock();
    }

    // Copies the pieces, which are in order of their chunks 0 .. nchunks - 1,
    // each with at least one piece. On the calling thread, in order:
    // open(c, wait) says whether chunk c may be copied now (wait: blocks until
    // it may), asked only once chunk c - depth is done; done(c) follows its last
    // piece. An exception from either ends the copy and is passed on.
    template <class Open, class Done>
    void run(const std::vector<Piece>& pieces, int nchunks, int depth, Open&& open, Done&& done) {
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
        const auto job = std::make_shared<Job>(pieces, nchunks);
        post(job);
        int opened = 0;
        try {
            for (int c = 0; c < nchunks; c++) {
                while (job->left[c].load(std::memory_order_acquire) > 0) {
                    while (opened < std::min(nchunks, c + depth) && open(opened, opened <= c)) job->open(++opened);
                    if (!job->copy_next()) std::this_thread::yield();
                }
                done(c);
            }
        } catch (...) {
            job->drain();
            post(nullptr);
            throw;
        }
        post(nullptr);
    }

private:
    // One copy. The helpers share it with the caller and may leave it after the
    // caller has: no piece is in flight by then.
    struct Job {
        const std::vector<Piece> pieces;
        std::unique_ptr<std::atomic<int>[]> left;  // pieces of each chunk still to be copied
        std::atomic<int> next{0}, copied{0}, opened{0};
        std::mutex mu;  // of the sleeping helpers
        std::condition_variable more;
        bool over = false;
        Job(const std::vector<Piece>& p, int nchunks) : pieces(p), left(new std::atomic<int>[nchunks]) {
            for (int c = 0; c < nchunks; c++) left[c].store(0, std::memory_order_relaxed);
            for (const Piece& q : p) left[q.chunk].fetch_add(1, std::memory_order_relaxed);
        }
        // copies the next piece, if there is one and its chunk is open
        bool copy_next() {
            int i = next.load(std::memory_order_relaxed);
            do {
                if (i >= (int)pieces.size() || pieces[i].chunk >= opened.load(std::memory_order_acquire)) return false;
            } while (!next.compare_exchange_weak(i, i + 1));
            copy(pieces[i]);
            left[pieces[i].chunk].fetch_sub(1, std::memory_order_release);
            copied.fetch_add(1, std::memory_order_release);
            return true;
        }
        void open(int n) {
            {
                std::lock_guard<std::mutex> lk(mu);
                opened.store(n, std::memory_order_release);
            }
            more.notify_all();
        }
        // takes the pieces away that nobody has begun, and waits for the others
        void drain() {
            const int begun = std::min(next.exchange((int)pieces.size()), (int)pieces.size());
            while (copied.load(std::memory_order_acquire) < begun) std::this_thread::yield();
        }
        void end() {
            {
                std::lock_guard<std::mutex> lk(mu);
                over = true;
            }
            more.notify_all();
        }
        // A helper: the pieces of open chunks, asleep while there are none. It
        // takes none before its chunk is open, so that nobody waits for a helper
        // to wake. (Helpers that waited by yielding kept three CPUs busy while the
        // caller waited for the link.)
        void help() {
            for (;;) {
                const int seen = opened.load(std::memory_order_acquire);
                while (copy_next()) {}
                std::unique_lock<std::mutex> lk(mu);
                more.wait(lk, [&] { return over || opened.load(std::memory_order_relaxed) != seen; });
                if (over) return;
            }
        }
    };

    static void copy(const Piece& p) {
        for (int r = 0; r < p.rows; r++)
            std::memcpy(p.dst + (int64_t)r * p.dst_stride, p.src + (int64_t)r * p.src_stride, p.bytes);
    }

    // the job helpers may join, in place of the one before
    void post(std::shared_ptr<Job> j) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            job_.swap(j);
            if (job_) gen_++;
        }
        if (j) j->end();
        else go_.notify_all();
    }

    void helper() {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lk(mu_);
        for (;;) {
            go_.wait(lk, [&] { return stop_ || (job_ && gen_ != seen); });
            if (stop_) return;
            seen = gen_;
            std::shared_ptr<Job> j = job_;
            lk.unlock();
            j->help();
            j.reset();
            lk.lock();
        }
    }

    std::vector<std::thread> threads_;
    std::mutex use_;  // held by the copy that has the helpers
    std::mutex mu_;
    std::condition_variable go_;
    std::shared_ptr<Job> job_;
    uint64_t gen_ = 0;
    bool stop_ = false;
};

}  // namespace vship
