// Locality order of TOR events on the device (locality.hip).
#pragma once

#include "tor_core.h"

namespace srfx {

// The buckets of a set's events and each bucket's next free place: a kernel
// over the events puts event e at place atomicAdd(&cursor[key[e]], 1), where
// neighbouring places hold near and nearly parallel tubes (order within a
// bucket arbitrary), subset [k n / K, (k + 1) n / K) to places of that range.
struct LocalityOrder {
    const int *key;
    unsigned *cursor;
};

// Workspace bytes of the order of n events in K subsets.
size_t locality_bytes(int64_t n, int64_t K);

// The order of the events of p in K subsets, in the workspace ws of
// locality_bytes(p.n, K).
int locality_order(const TorParams &p, int64_t K, LocalityOrder &order, char *ws, hipStream_t st);

// place[e] = the place of event e.
int locality_places(const TorParams &p, int64_t K, int *place, char *ws, hipStream_t st);

} // namespace srfx
