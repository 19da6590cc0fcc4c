// What tests change inside a handle, to reach code that no call of theirs
// would: built with the library's own headers, on its device memory.
#include "batch.hpp"
#include "internal.hpp"

namespace {

int put(void *device, const void *host, size_t bytes) {
    return hipMemcpy(device, host, bytes, hipMemcpyHostToDevice) == hipSuccess ? 0 : 1;
}

}  // namespace

extern "C" {

// As if v look-backs of the radix sort had given up (the handle is idle).
int access_sort_stall(gsim_sim *s, uint32_t v) { return put(&s->bh.ctr->sort_stall, &v, 4); }
int access_batch_sort_stall(gsim_batch *b, uint32_t v) {
    return put(&b->d.counts->sort_stall, &v, 4);
}

// Walks address nodes by slot from this many on.
void access_narrow_nodes(gsim_sim *s, size_t n) { s->narrow_nodes = n; }
void access_batch_narrow_nodes(gsim_batch *b, size_t n) {
    b->narrow_nodes = n;
    b->dirty = true;
}

}  // extern "C"
