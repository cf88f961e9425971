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
// exact size and not kept.  The cache is bounded (kPoolCap: the largest blocks
// are given back first) and given back whole when the device runs out of memory
// (dev_alloc retries) and at shutdown; blocks of another device are never
// reused.
#include <map>
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
struct Pool {
    std::unordered_map<void *, Block> blocks;  // every live or cached block
    std::map<int, std::vector<void *>> free_lists;
    size_t cached = 0;
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

}  // namespace

void pool_trim() {
    std::lock_guard<std::recursive_mutex> lock(api_mutex());
    Pool &P = pool();
    for (auto &l : P.free_lists)
        for (void *p : l.second) {
            P.blocks.erase(p);
            (void)hipFree(p);  // waits for the work that still uses it
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
        *p = it->second.back();
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
        for (auto l = P.free_lists.rbegin(); P.cached + n > kPoolCap && l != P.free_lists.rend(); ++l)
            while (P.cached + n > kPoolCap && !l->second.empty()) {
                void *q = l->second.back();
                l->second.pop_back();
                P.cached -= class_bytes(l->first);
                P.blocks.erase(q);
                dev_free(q);  // waits for the work that still uses it
            }
        try {
            P.free_lists[c].push_back(p);
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
