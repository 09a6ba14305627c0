/*
 * memory.hip - the per-context caching device allocator (see Pool in
 * bcmg_internal.h).
 */
#include "bcmg_internal.h"

#include <algorithm>

namespace bcmg {

namespace {
thread_local Pool *g_pool = nullptr;
}

Pool *current_pool() { return g_pool; }

PoolScope::PoolScope(Pool *p) : prev(g_pool) { g_pool = p; }
PoolScope::~PoolScope() { g_pool = prev; }

size_t Pool::size_class(size_t bytes)
{
    if (bytes <= 4096) return (bytes + 255) & ~(size_t)255;
    int e = 63 - __builtin_clzll((unsigned long long)bytes);
    const size_t step = (size_t)1 << (e - 2);
    return (bytes + step - 1) & ~(step - 1);
}

namespace {
void *device_block(size_t bytes)
{
    void *p = nullptr;
    if (hipMalloc(&p, bytes) == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
}
} // namespace

/* the next cls bytes of a chunk that has them, or of a new one (null: the
   device has no room for a chunk) */
void *Pool::cut(size_t cls, Chunk **from)
{
    Chunk *c = nullptr;
    size_t last = 0;
    for (Chunk &k : chunks_) {
        last = std::max(last, k.size);
        if (!c && k.size - k.used >= cls) c = &k;
    }
    if (!c) {
        const size_t want = std::max(cls, std::min(CHUNK_MAX, std::max(CHUNK_MIN, 2 * last)));
        char *base = static_cast<char *>(device_block(want));
        if (!base) return nullptr;
        try {
            chunks_.emplace_back();
        } catch (...) {
            (void)hipFree(base);
            throw;
        }
        c = &chunks_.back();
        c->base = base;
        c->size = want;
    }
    void *p = c->base + c->used;
    c->used += cls;
    *from = c;
    return p;
}

void *Pool::alloc(size_t bytes)
{
    const size_t cls = size_class(bytes);
    void *p = nullptr;
    Chunk *from = nullptr;
    auto it = free_.lower_bound(cls);
    const auto end = free_.upper_bound(cls);
    while (own_blocks && it != end && it->second.second) ++it;
    if (it != end) {
        p = it->second.first;
        from = it->second.second;
        free_.erase(it);
        cached -= cls;
    } else {
        for (int attempt = 0; !p && attempt < 2; attempt++) {
            if (attempt) trim();
            if (cls <= SUB_MAX && !own_blocks) p = cut(cls, &from);
            if (!p) p = device_block(cls);
        }
        if (!p)
            throw Error(BCMG_ENOMEM, "device allocation of " + std::to_string(cls) +
                                         " bytes failed");
    }
    cls_[p] = Block{cls, from};
    if (from) from->out++;
    live += cls;
    return p;
}

void Pool::release(void *p)
{
    auto it = cls_.find(p);
    if (it == cls_.end()) {
        (void)hipFree(p);
        return;
    }
    const Block b = it->second;
    cls_.erase(it);
    live -= b.cls;
    if (free_released && !b.chunk) {
        (void)hipFree(p);
        return;
    }
    free_.emplace(b.cls, std::make_pair(p, b.chunk));
    cached += b.cls;
    if (b.chunk && --b.chunk->out == 0 && free_released) free_chunks();
}

/* give back the chunks none of whose blocks are out (hipFree waits for the
   work that used them) */
void Pool::free_chunks()
{
    for (auto it = free_.begin(); it != free_.end();) {
        if (it->second.second && it->second.second->out == 0) {
            cached -= it->first;
            it = free_.erase(it);
        } else {
            ++it;
        }
    }
    for (auto it = chunks_.begin(); it != chunks_.end();) {
        if (it->out == 0) {
            (void)hipFree(it->base);
            it = chunks_.erase(it);
        } else {
            ++it;
        }
    }
}

void Pool::trim()
{
    if (!free_.empty() || !chunks_.empty()) (void)hipDeviceSynchronize();
    for (auto it = free_.begin(); it != free_.end();) {
        if (!it->second.second) {
            (void)hipFree(it->second.first);
            cached -= it->first;
            it = free_.erase(it);
        } else {
            ++it;
        }
    }
    free_chunks();
}

Pool::~Pool() { trim(); }

void *dev_alloc(Pool *pool, size_t bytes)
{
    if (pool) return pool->alloc(bytes);
    void *p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) {
        (void)hipGetLastError();
        throw Error(BCMG_ENOMEM, "device allocation of " + std::to_string(bytes) + " bytes failed");
    }
    return p;
}

void dev_free(Pool *pool, void *p)
{
    if (!p) return;
    if (pool)
        pool->release(p);
    else
        (void)hipFree(p);
}

} // namespace bcmg
