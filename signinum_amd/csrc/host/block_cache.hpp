// Memory blocks kept for reuse instead of freed.
#pragma once
#include <algorithm>
#include <cstdint>
#include <iterator>
#include <map>
#include <unordered_map>

namespace sgn {

// get() hands out a cached block of at least `bytes` (at most twice that,
// plus 1 MiB) or allocates one; put() caches it, freeing the largest cached
// blocks while more than `cap` bytes are cached.  An allocation that fails is
// tried once more after the cache and its sibling (null: none) have given back
// what they hold.  Not thread-safe: one owner drives a cache and its sibling.
// M: alloc(void **, uint64_t) returns 0 or an error code, free(void *).
template <class M>
class BlockCache {
  public:
    explicit BlockCache(uint64_t cap, BlockCache *sibling = nullptr) : cap_(cap), sibling_(sibling) {}
    ~BlockCache() { trim(0); }
    BlockCache(const BlockCache &) = delete;
    BlockCache &operator=(const BlockCache &) = delete;
    int get(uint64_t bytes, void **out) {
        bytes = std::max<uint64_t>(bytes, 256);
        auto it = free_.lower_bound(bytes);
        if (it != free_.end() && it->first <= 2 * bytes + (uint64_t(1) << 20)) {
            *out = it->second;
            size_[*out] = it->first;
            cached_ -= it->first;
            free_.erase(it);
            return 0;
        }
        const int e = alloc(bytes, out);
        if (!e) size_[*out] = bytes;
        return e;
    }
    void put(void *p) {
        if (!p) return;
        const auto it = size_.find(p);
        if (it == size_.end()) return;
        free_.emplace(it->second, p);
        cached_ += it->second;
        size_.erase(it);
        trim(cap_);
    }
    // Memory that the cache does not keep, with the same second try.
    int alloc(uint64_t bytes, void **out) {
        int e = M::alloc(out, bytes);
        if (e && (cached_ || (sibling_ && sibling_->cached_))) {
            trim(0);
            if (sibling_) sibling_->trim(0);
            e = M::alloc(out, bytes);
        }
        return e;
    }
    uint64_t cached() const { return cached_; }
    void set_sibling(BlockCache *c) { sibling_ = c; }

  private:
    void trim(uint64_t keep) {
        while (cached_ > keep && !free_.empty()) {
            auto last = std::prev(free_.end());
            M::free(last->second);
            cached_ -= last->first;
            free_.erase(last);
        }
    }
    uint64_t cap_, cached_ = 0;
    BlockCache *sibling_;
    std::multimap<uint64_t, void *> free_;        // cached: size -> block
    std::unordered_map<void *, uint64_t> size_;  // handed out: block -> size
};

}  // namespace sgn
