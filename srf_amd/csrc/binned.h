// Binned forms of the untiled TOR scatters (binned.hip), for the entry points
// of tor.hip.
#pragma once

#include "tor_core.h"

namespace srfx {

// Whether an untiled scatter of p.n events runs binned by its size and flags, and
// whether it may on stream st.
bool binned_rule(const TorParams &p, uint32_t flags);
bool binned_ok(const TorParams &p, uint32_t flags, hipStream_t st);

// The untiled scatters kBack, kMap, kAdj (p.val, p.out, output strides set)
// and the OSEM pass kOsem (p.img as well) over p's events, binned into image
// tiles on the device.  *done is set when the work was enqueued; else nothing
// was and the caller runs the direct kernels.
int binned_scatter(int mode, const TorParams &p, hipStream_t st, bool *done);

// The untiled projection (p.img, p.out set) of a large event set in locality
// order.  done as above.
int sorted_project(const TorParams &p, uint32_t flags, hipStream_t st, bool *done);

} // namespace srfx
