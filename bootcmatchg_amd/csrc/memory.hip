/*
 * memory.hip - the per-context caching device allocator (see Pool in
 * bcmg_internal.h).
 */
#include "bcmg_internal.h"

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

/* a cached allocation of its own of that class, or null */
void *Pool::cached(size_t cls)
{
    const auto it = free_.find(cls);
    if (it == free_.end()) return nullptr;
    void *const p = it->second;
    free_.erase(it);
    return p;
}

/* cls bytes of a new chunk (null: the device has no room for one) */
void *Pool::cut(size_t cls)
{
    const size_t size = chunks_.next_size(cls);
    char *const base = static_cast<char *>(device_block(size));
    if (!base) return nullptr;
    try {
        chunks_.add(base, size);
    } catch (...) {
        (void)hipFree(base);
        throw;
    }
    return chunks_.take(cls);
}

void *Pool::alloc(size_t bytes)
{
    const size_t cls = size_class(bytes);
    const bool small = cls <= Chunks::SUB_MAX && !own_blocks;
    Block b{cls, true};
    void *p = small ? chunks_.take(cls) : nullptr;
    if (!p && (p = cached(cls))) b.cut = false;
    for (int attempt = 0; !p && attempt < 2; attempt++) {
        if (attempt) trim();
        if (small) p = cut(cls);
        if (!p && (p = device_block(cls))) b.cut = false;
    }
    if (!p)
        throw Error(BCMG_ENOMEM,
                    "device allocation of " + std::to_string(cls) + " bytes failed");
    cls_[p] = b;
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
    if (b.cut) {
        if (chunks_.give(static_cast<char *>(p), b.cls) && free_released) free_chunks();
    } else if (free_released) {
        (void)hipFree(p);
    } else {
        free_.emplace(b.cls, p);
    }
}

/* give back the chunks none of whose blocks are out (hipFree waits for the
   work that used them) */
void Pool::free_chunks()
{
    for (char *base : chunks_.take_whole()) (void)hipFree(base);
}

void Pool::trim()
{
    if (!free_.empty() || !chunks_.empty()) (void)hipDeviceSynchronize();
    for (auto &kv : free_) (void)hipFree(kv.second);
    free_.clear();
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
