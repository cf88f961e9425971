// Storage of the op-level API: device blocks kept for reuse.
//
// Every op returns new storage and the caller frees it (the reference's
// functional style), so one layer run op by op allocates and frees about 40
// blocks.  hipMalloc plus a synchronising hipFree cost 7 us a pair for small
// blocks and up to 1 ms for tens of MB, and kept the host from running ahead
// of the stream: a 130-row 8B MLP spent 2.7 of 2.9 ms there, a 512-token 8B
// layer 6.5 of 7.4 ms.
//
// All op work runs on the context's one stream, so a block freed by the host
// is handed to a later op in stream order without waiting.  Blocks up to
// kPoolMax are filed by size class (8 per power of two) under the API lock;
// larger ones, and blocks whose class finds no memory, are allocated at their
// exact size and not kept.  The cache is bounded (kPoolCap: the blocks unused for
// longest are given back first, so that what a program no longer needs does not
// push out what it uses) and given back whole when the device runs out of
// memory (dev_alloc retries) and at shutdown; blocks of another device are never
// reused.
#include <new>
#include <unordered_map>

#include "internal.h"

namespace scry {
namespace {

constexpr size_t kPoolCap = (size_t)2 << 30;  // under 1% of the card's memory
constexpr size_t kPoolMax = kPoolCap / 2;

struct Block {
    int cls, device;
};
struct Free {
    void *p;
    uint64_t when;  // number of the free
};
struct Pool {
    std::unordered_map<void *, Block> blocks;  // every live or cached block
    std::unordered_map<int, std::vector<Free>> free_lists;  // by class, oldest first
    size_t cached = 0;
    uint64_t frees = 0;
};
Pool &pool() {
    static Pool *p = new Pool;  // never destroyed: storage may be freed during process exit
    return *p;
}

// class c holds blocks of (8 + c % 8) << (c / 8 + 5) bytes: 256, 288, ...
size_t class_bytes(int c) { return (size_t)(8 + c % 8) << (c / 8 + 5); }
int class_of(size_t bytes) {
    if (bytes <= 256) return 0;
    int e = 0;
    while (((bytes - 1) >> (e + 5)) >= 16) e++;
    return 8 * e + (int)((bytes - 1) >> (e + 5)) - 8 + 1;
}

// (P.cached > 0)
void give_back_oldest(Pool &P) {
    auto old = P.free_lists.end();
    for (auto l = P.free_lists.begin(); l != P.free_lists.end(); ++l)
        if (!l->second.empty() && (old == P.free_lists.end() || l->second[0].when < old->second[0].when)) old = l;
    void *p = old->second[0].p;
    old->second.erase(old->second.begin());
    P.cached -= class_bytes(old->first);
    P.blocks.erase(p);
    dev_free(p);  // waits for the work that still uses it
}

}  // namespace

void pool_trim() {
    std::lock_guard<std::recursive_mutex> lock(api_mutex());
    Pool &P = pool();
    for (auto &l : P.free_lists)
        for (const Free &f : l.second) {
            P.blocks.erase(f.p);
            dev_free(f.p);  // waits for the work that still uses it
        }
    P.free_lists.clear();
    P.cached = 0;
}

int pool_alloc(void **p, size_t bytes) {
    std::lock_guard<std::recursive_mutex> lock(api_mutex());
    *p = nullptr;
    if (bytes > kPoolMax) return dev_alloc(p, bytes);
    Pool &P = pool();
    const int c = class_of(bytes);
    auto it = P.free_lists.find(c);
    if (it != P.free_lists.end() && !it->second.empty()) {
        *p = it->second.back().p;
        it->second.pop_back();
        P.cached -= class_bytes(c);
        return SCRY_OK;
    }
    const int rc = dev_alloc(p, class_bytes(c));
    if (rc == SCRY_ERR_OOM) return dev_alloc(p, bytes);
    if (rc) return rc;
    try {
        P.blocks[*p] = Block{c, ctx().device};
    } catch (const std::bad_alloc &) {  // not filed: freed as it is
    }
    return SCRY_OK;
}

void pool_free(void *p) {
    if (!p) return;
    std::lock_guard<std::recursive_mutex> lock(api_mutex());
    Pool &P = pool();
    auto it = P.blocks.find(p);
    if (it != P.blocks.end() && ctx().init && it->second.device == ctx().device) {
        const int c = it->second.cls;
        const size_t n = class_bytes(c);
        while (P.cached + n > kPoolCap) give_back_oldest(P);
        try {
            P.free_lists[c].push_back(Free{p, P.frees++});
            P.cached += n;
            return;
        } catch (const std::bad_alloc &) {
        }
    }
    if (it != P.blocks.end()) P.blocks.erase(it);
    if (ctx().init) (void)hipStreamSynchronize(ctx().stream);
    dev_free(p);
}

}  // namespace scry
