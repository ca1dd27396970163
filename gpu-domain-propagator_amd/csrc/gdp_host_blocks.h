// gdp_host_blocks.h - pinned host blocks that outlive one problem.  Plain C++,
// no HIP (the allocation is the caller's): tested on the CPU.
#pragma once

#include <cstddef>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace gdp {

// Pinned host blocks for launch tables, outcomes and small bound vectors, by
// powers of two from 4 KiB.  Freed blocks of up to 1 MiB are kept for the next
// request, 16 MiB in all; the others go back to the runtime.
class HostBlocks {
  public:
    // alloc throws when there is no memory
    HostBlocks(void *(*alloc)(size_t), void (*release)(void *)) : alloc_(alloc), release_(release) {}

    void *take(size_t bytes, size_t *size) {
        size_t want = 4096;
        while (want < bytes) want *= 2;
        {
            std::lock_guard<std::mutex> lk(mu_);
            auto it = free_.find(want);
            if (it != free_.end() && !it->second.empty()) {
                void *p = it->second.back();
                it->second.pop_back();
                kept_ -= want;
                *size = want;
                return p;
            }
        }
        void *p = alloc_(want);
        *size = want;
        return p;
    }
    void give(void *p, size_t size) {
        if (!p) return;
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (size <= (1u << 20) && kept_ + size <= (16u << 20)) {
                free_[size].push_back(p);
                kept_ += size;
                return;
            }
        }
        release_(p);
    }

  private:
    void *(*alloc_)(size_t);
    void (*release_)(void *);
    std::mutex mu_;
    std::unordered_map<size_t, std::vector<void *>> free_;
    size_t kept_ = 0;
};

// A pinned block of at least the bytes last asked for.
struct HostBlock {
    HostBlocks &pool;
    char *p = nullptr;
    size_t size = 0;  // 0 without a block, also after a request that failed

    explicit HostBlock(HostBlocks &from) : pool(from) {}
    HostBlock(const HostBlock &) = delete;
    HostBlock &operator=(const HostBlock &) = delete;
    ~HostBlock() { pool.give(p, size); }

    char *get(size_t bytes) {
        if (bytes > size) {
            pool.give(p, size);
            p = nullptr;
            size = 0;
            p = static_cast<char *>(pool.take(bytes, &size));
        }
        return p;
    }
};

}  // namespace gdp
