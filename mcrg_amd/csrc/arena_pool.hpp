// Device memory of the library: allocations, and the one arena that a context
// keeps between servers.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <vector>

namespace mcrg {

// The job arena of the context's server that was destroyed last, for the next
// one of the same size: device memory that is freed has to be cleared by the
// driver (about 100 ms for 4 GiB) before it can be allocated again, and once all
// of the device's memory has been through a process's hands every new arena
// waits for that.  At most one arena of at most kMaxBytes a context, the newest
// in place of an older one.  It is freed with the context and the last of its
// servers, and when an allocation of the library on the same device, whatever
// the context, finds no memory (device_malloc).
class ArenaPool {
  public:
    static constexpr size_t kMaxBytes = size_t(4) << 30;

    explicit ArenaPool(int device) : device_(device)
    {
        std::lock_guard<std::mutex> lock(all_mu_);
        all().push_back(this);
    }
    ~ArenaPool()
    {
        {
            std::lock_guard<std::mutex> lock(all_mu_);
            all().erase(std::remove(all().begin(), all().end(), this), all().end());
        }
        (void)drop();
    }
    ArenaPool(const ArenaPool &) = delete;
    ArenaPool &operator=(const ArenaPool &) = delete;

    // The kept arena if it has this size, else null.
    void *take(size_t bytes)
    {
        std::lock_guard<std::mutex> lock(mu_);
        if (!base_ || bytes_ != bytes) return nullptr;
        void *p = base_;
        base_ = nullptr;
        return p;
    }
    // False when the caller has to free it.  Nothing may read or write it any more.
    bool give(void *base, size_t bytes)
    {
        if (bytes > kMaxBytes) return false;
        void *old;
        {
            std::lock_guard<std::mutex> lock(mu_);
            old = base_;
            base_ = base;
            bytes_ = bytes;
        }
        if (old) (void)hipFree(old);
        return true;
    }
    // Frees the arenas that the contexts of `device` keep; whether there were any.
    static bool drop_all(int device)
    {
        std::lock_guard<std::mutex> lock(all_mu_);
        bool any = false;
        for (ArenaPool *p : all())
            if (p->device_ == device) any = p->drop() || any;
        return any;
    }

  private:
    bool drop()
    {
        std::lock_guard<std::mutex> lock(mu_);
        if (!base_) return false;
        (void)hipFree(base_);
        base_ = nullptr;
        return true;
    }

    const int device_;
    std::mutex mu_;
    void *base_ = nullptr;
    size_t bytes_ = 0;

    // every pool of the process; never destroyed, since contexts may outlive
    // static objects
    static std::vector<ArenaPool *> &all()
    {
        static auto *v = new std::vector<ArenaPool *>;
        return *v;
    }
    static inline std::mutex all_mu_;
};

// hipMalloc on the current device, which may have idle arenas to give up first.
template <typename T>
hipError_t device_malloc(T **p, size_t bytes)
{
    void *v = nullptr;
    hipError_t e = hipMalloc(&v, bytes);
    if (e == hipErrorOutOfMemory) {
        int device = 0;
        if (hipGetDevice(&device) == hipSuccess && ArenaPool::drop_all(device)) {
            (void)hipGetLastError();
            e = hipMalloc(&v, bytes);
        }
    }
    *p = e == hipSuccess ? static_cast<T *>(v) : nullptr;
    return e;
}

// Makes room for `count` items in the table p of cap items, at least twice what
// it had when it has to move; its contents go.  Without memory there is no table.
template <typename T>
hipError_t device_regrow(T *&p, size_t &cap, size_t count)
{
    if (count <= cap) return hipSuccess;
    const size_t want = std::max(count, 2 * cap);
    if (p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
    const hipError_t e = device_malloc(&p, sizeof(T) * want);
    if (e == hipSuccess) cap = want;
    return e;
}

}  // namespace mcrg
