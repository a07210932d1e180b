// Host interface of the persistent decode kernel for shapes that decode_persistent.hip has no instantiation of.
#ifndef WGPT_DECODE_GENERIC_H
#define WGPT_DECODE_GENERIC_H

#include "decode_persistent.h"

namespace wgpt {

constexpr int DG_SPLIT = 8;  // most slices of the context per head

// Shapes that launch_decode_generic takes.
bool decode_generic_supports(int d, int H, int hs, int ctx, int V, int compute_units);
// a.nsteps steps, greedy or sampled as a.top_k says; a.colparams is not used. Epochs as persistent_epochs_per_step says.
hipError_t launch_decode_generic(const PersistentArgs& a, hipStream_t s);

}  // namespace wgpt

#endif
