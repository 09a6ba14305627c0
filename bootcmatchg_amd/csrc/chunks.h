/*
 * chunks.h - the space of a pool's chunks: which bytes are free, which are out.
 * Holds addresses only (no HIP): the pool gets and gives back the memory.
 */
#pragma once

#include <algorithm>
#include <cstddef>
#include <map>
#include <set>
#include <unordered_map>
#include <utility>
#include <vector>

namespace bcmg {

/* A block that comes back is kept for the next one of its size; where none of
   that size is kept and no free range of a chunk holds the block, the kept ones
   join their free neighbours first. So a chunk serves blocks of any size over
   and over, and a set-up, which asks for some sizes hundreds of times, cuts and
   joins seldom (0.06 us an operation; 0.37 with a join each time, which a
   smoothed 39^3 set-up and solve paid with 7.6 ms instead of 7.45). */
class Chunks {
  public:
    /* longest block cut from a chunk; a new chunk's size is twice the largest
       so far between the two limits */
    static constexpr size_t SUB_MAX = (size_t)16 << 20;
    static constexpr size_t CHUNK_MIN = (size_t)8 << 20, CHUNK_MAX = (size_t)32 << 20;

    size_t total() const { return total_; }   /* bytes of all chunks */
    size_t free() const { return free_bytes_; }
    bool empty() const { return chunks_.empty(); }

    /* a block of `bytes`, or null where no chunk has room */
    char *take(size_t bytes)
    {
        char *p = nullptr;
        const auto k = kept_.find(bytes);
        if (k != kept_.end() && !k->second.empty()) {
            p = k->second.back();
            k->second.pop_back();
        } else {
            p = cut(bytes);
            if (!p && join_kept()) p = cut(bytes);
            if (!p) return nullptr;
        }
        free_bytes_ -= bytes;
        chunk_of(p)->second.out++;
        return p;
    }

    /* the size of the chunk to add for a block of `bytes` */
    size_t next_size(size_t bytes) const
    {
        size_t last = 0;
        for (const auto &c : chunks_) last = std::max(last, c.second.size);
        return std::max(bytes, std::min(CHUNK_MAX, std::max(CHUNK_MIN, 2 * last)));
    }

    void add(char *base, size_t bytes)
    {
        chunks_.emplace(base, Chunk{bytes, 0});
        total_ += bytes;
        free_bytes_ += bytes;
        put(base, bytes);
    }

    /* a block back; true when its chunk has no block out any more */
    bool give(char *p, size_t bytes)
    {
        kept_[bytes].push_back(p);
        free_bytes_ += bytes;
        return --chunk_of(p)->second.out == 0;
    }

    /* forget the chunks that have no block out; their addresses */
    std::vector<char *> take_whole()
    {
        join_kept();
        std::vector<char *> out;
        for (auto c = chunks_.begin(); c != chunks_.end();) {
            if (c->second.out > 0) {
                ++c;
                continue;
            }
            out.push_back(c->first);
            total_ -= c->second.size;
            free_bytes_ -= c->second.size;
            drop(free_.find(c->first));
            c = chunks_.erase(c);
        }
        return out;
    }

  private:
    struct Chunk {
        size_t size, out;   /* bytes; blocks out */
    };
    using Ranges = std::map<char *, size_t>;
    std::map<char *, Chunk> chunks_;                /* by address */
    Ranges free_;                                   /* free ranges by address */
    std::set<std::pair<size_t, char *>> by_size_;   /* the same by size */
    std::unordered_map<size_t, std::vector<char *>> kept_;   /* blocks back, by size */
    size_t total_ = 0, free_bytes_ = 0;

    std::map<char *, Chunk>::iterator chunk_of(char *p)
    {
        return std::prev(chunks_.upper_bound(p));
    }
    void put(char *p, size_t bytes)
    {
        free_.emplace(p, bytes);
        by_size_.emplace(bytes, p);
    }
    Ranges::iterator drop(Ranges::iterator f)
    {
        by_size_.erase({f->second, f->first});
        return free_.erase(f);
    }

    /* the front of the shortest free range that holds a block */
    char *cut(size_t bytes)
    {
        const auto s = by_size_.lower_bound({bytes, nullptr});
        if (s == by_size_.end()) return nullptr;
        char *const p = s->second;
        const size_t rest = s->first - bytes;
        drop(free_.find(p));
        if (rest) put(p + bytes, rest);
        return p;
    }

    /* the kept blocks into the free ranges; whether there were any */
    bool join_kept()
    {
        bool any = false;
        for (auto &k : kept_) {
            for (char *p : k.second) join(p, k.first);
            any = any || !k.second.empty();
            k.second.clear();
        }
        return any;
    }
    void join(char *p, size_t bytes)
    {
        const auto c = chunk_of(p);
        auto next = free_.lower_bound(p);
        if (next != free_.end() && next->first == p + bytes &&
            p + bytes != c->first + c->second.size) {
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
    }
};

} // namespace bcmg
