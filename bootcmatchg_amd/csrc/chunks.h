/*
 * chunks.h - the space of a pool's chunks: which bytes are free, which are out.
 * Holds addresses only (no HIP): the pool gets and gives back the memory.
 */
#pragma once

#include <algorithm>
#include <cstddef>
#include <map>
#include <set>
#include <utility>
#include <vector>

namespace bcmg {

/* A block is cut from the shortest free range that holds it, and joins its free
   neighbours in the chunk when it comes back, so a chunk serves blocks of any
   size over and over. */
class Chunks {
  public:
    /* longest block cut from a chunk; a new chunk's size is twice the largest
       so far between the two limits */
    static constexpr size_t SUB_MAX = (size_t)16 << 20;
    static constexpr size_t CHUNK_MIN = (size_t)8 << 20, CHUNK_MAX = (size_t)32 << 20;

    size_t total() const { return total_; }   /* bytes of all chunks */
    size_t free() const { return free_bytes_; }
    bool empty() const { return chunks_.empty(); }

    /* a block of `bytes`, or null where no free range holds it */
    char *take(size_t bytes)
    {
        const auto s = by_size_.lower_bound({bytes, nullptr});
        if (s == by_size_.end()) return nullptr;
        char *const p = s->second;
        const size_t rest = s->first - bytes;
        drop(free_.find(p));
        if (rest) put(p + bytes, rest);
        return p;
    }

    /* the size of the chunk to add for a block of `bytes` */
    size_t next_size(size_t bytes) const
    {
        size_t last = 0;
        for (const auto &c : chunks_) last = std::max(last, c.second);
        return std::max(bytes, std::min(CHUNK_MAX, std::max(CHUNK_MIN, 2 * last)));
    }

    void add(char *base, size_t bytes)
    {
        chunks_.emplace(base, bytes);
        total_ += bytes;
        put(base, bytes);
    }

    /* a block back; true when its chunk has no block out any more */
    bool give(char *p, size_t bytes)
    {
        const auto c = std::prev(chunks_.upper_bound(p));
        auto next = free_.lower_bound(p);
        if (next != free_.end() && next->first == p + bytes && p + bytes != c->first + c->second) {
            bytes += next->second;
            next = drop(next);
        }
        if (next != free_.begin() && p != c->first) {
            const auto prev = std::prev(next);
            if (prev->first + prev->second == p) {
                p = prev->first;
                bytes += prev->second;
                drop(prev);
            }
        }
        put(p, bytes);
        return p == c->first && bytes == c->second;
    }

    /* forget the chunks that have no block out; their addresses */
    std::vector<char *> take_whole()
    {
        std::vector<char *> out;
        for (auto c = chunks_.begin(); c != chunks_.end();) {
            const auto f = free_.find(c->first);
            if (f == free_.end() || f->second != c->second) {
                ++c;
                continue;
            }
            out.push_back(c->first);
            total_ -= c->second;
            drop(f);
            c = chunks_.erase(c);
        }
        return out;
    }

  private:
    using Ranges = std::map<char *, size_t>;
    Ranges chunks_, free_;                          /* by address */
    std::set<std::pair<size_t, char *>> by_size_;   /* the free ranges */
    size_t total_ = 0, free_bytes_ = 0;

    void put(char *p, size_t bytes)
    {
        free_.emplace(p, bytes);
        by_size_.emplace(bytes, p);
        free_bytes_ += bytes;
    }
    Ranges::iterator drop(Ranges::iterator f)
    {
        by_size_.erase({f->second, f->first});
        free_bytes_ -= f->second;
        return free_.erase(f);
    }
};

} // namespace bcmg
