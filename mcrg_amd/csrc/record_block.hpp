// Records of a batch's jobs read ahead.  One job's records cost a round trip to
// the device (26 us); a caller that reads one job after the other gets the
// following ones along, more with every such read, in one copy (4096 jobs: 110
// -> 12 ms with the callers' own time).
//
// Calls on one batch may come from several threads.  A block is only kept
// between runs: while a run is in progress every read goes to the device, and
// both ends of a run drop what was read before.  So a read gives what a single
// read at its place would.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

namespace mcrg {

class RecordBlock {
  public:
    static constexpr size_t kMaxBytes = size_t(1) << 20;
    static constexpr int kMaxJobs = 4096;

    // Held while the batch runs.
    class Running {
      public:
        explicit Running(RecordBlock &b) : b_(b) { b_.run(1); }
        ~Running() { b_.run(-1); }
        Running(const Running &) = delete;
        Running &operator=(const Running &) = delete;

      private:
        RecordBlock &b_;
    };

    // The `bytes` of records of `job` to host; E(0) is success.
    //   more(k)             bytes that job job + k adds to a block that starts
    //                       with job, 0 where it cannot be part of one
    //   one()               a single read of the job to host
    //   block(n, off, data) jobs job .. job + n - 1 to data (resized), off[k]
    //                       where each begins; off left empty: no such block
    template <typename E, typename More, typename One, typename Block>
    E read(int job, char *host, size_t bytes, More more, One one, Block block)
    {
        std::unique_lock<std::mutex> lk(mu_);
        if (running_ > 0) {
            lk.unlock();
            return one();
        }
        if (job >= first_ && job < first_ + count_) {
            std::memcpy(host, data_.data() + off_[(size_t)(job - first_)], bytes);
            next_ = job + 1;
            return E(0);
        }
        window_ = job == next_ ? std::min(8 * window_, kMaxJobs) : 1;
        count_ = 0;
        next_ = job + 1;
        int n = 1;
        for (size_t total = bytes; n < window_; ++n) {
            const size_t add = more(n);
            if (add == 0 || total + add > kMaxBytes) break;
            total += add;
        }
        if (n == 1) return one();
        off_.clear();
        E e;
        try {
            e = block(n, off_, data_);
        } catch (const std::bad_alloc &) {
            return one();
        }
        if (e != E(0)) return e;
        if (off_.empty()) return one();
        first_ = job;
        count_ = n;
        std::memcpy(host, data_.data() + off_[0], bytes);
        return e;
    }

  private:
    void run(int by)
    {
        std::lock_guard<std::mutex> lk(mu_);
        running_ += by;
        count_ = 0;
        next_ = -1;
    }

    std::mutex mu_;
    std::vector<char> data_;
    std::vector<size_t> off_;   // per job, into data_
    int first_ = 0, count_ = 0;
    int next_ = -1, window_ = 1;  // the job behind the last one read, jobs then read at once
    int running_ = 0;             // runs in progress
};

}  // namespace mcrg
