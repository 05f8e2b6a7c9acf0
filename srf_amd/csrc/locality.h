// Locality order of TOR events on the device (locality.hip).
#pragma once

#include "tor_core.h"

namespace srfx {

// The buckets of a set's events and each bucket's next free place: a kernel
// over the events puts event e at place atomicAdd(&cursor[key[e]], 1), where
// neighbouring places hold near and nearly parallel tubes (order within a
// bucket arbitrary).
struct LocalityOrder {
    const int *key;
    unsigned *cursor;
};

// Workspace bytes of locality_order for n events.
size_t locality_bytes(int64_t n);

// The order of the events of p, in the workspace ws of locality_bytes(p.n).
int locality_order(const TorParams &p, LocalityOrder &order, char *ws, hipStream_t st);

} // namespace srfx
