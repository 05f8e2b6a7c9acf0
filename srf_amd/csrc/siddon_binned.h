// Binned forms of the untiled Siddon scatters (siddon_tile.hip), for the entry
// points of siddon.hip, and the set-up both share.
#pragma once

#include "siddon_core.h"

namespace srfx {

int siddon_setup(SidParams &p, const float *lors, int64_t n, int64_t ld, const srfx_grid &g,
                 float tof_bin, float tof_sigma2);

// Whether an untiled scatter of p.n rays runs binned by its size, and whether it
// may on stream st.
bool siddon_binned_rule(const SidParams &p);
bool siddon_binned_ok(const SidParams &p, hipStream_t st);

// The untiled scatters kBack, kMap, kAdj (p.val, p.out set) and the OSEM pass
// kOsem (p.img as well), binned into image tiles on the device: records and
// listings per piece of at most 2^19 rays in a stream-ordered workspace, no
// synchronisation.  *done is set when the work was enqueued; else nothing was
// and the caller runs the direct kernels.
int siddon_binned_scatter(int mode, const SidParams &p, hipStream_t st, bool *done);

} // namespace srfx
