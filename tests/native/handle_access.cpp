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

// The walk's launch order (`units` workgroups); 0 if there is a plan.
int access_order(gsim_sim *s, uint32_t *out, size_t units) {
    if (!s->bh.order_valid) return 1;
    return hipMemcpy(out, s->bh.order, sizeof(uint32_t) * units, hipMemcpyDeviceToHost) == hipSuccess
               ? 0
               : 2;
}

// Workgroups that take direct-sum blocks, and the blocks.
void access_batch_direct_sums(const gsim_batch *b, uint32_t *groups, uint32_t *blocks) {
    *groups = b->h_counts.ds_groups;
    *blocks = b->h_counts.n_ds;
}

}  // extern "C"
