// What the entry points of this library share beyond the public C ABI (include/flashlstm/lstm_core.h).
#pragma once
#include "../../include/flashlstm/lstm_core.h"
#include "pack.h"

namespace flstm_hip {

// flstm_core_pack_weights without the wait at its end: for callers whose next calls on the plan use the same stream.
int core_pack_weights_async(flstm_core_plan* plan, const float* w_ih, const float* w_hh, hipStream_t stream);

// Hands the next flstm_core_forward_steps (forward) or flstm_core_backward_steps call of the pass in progress copies to
// make beside its recurrence on workgroups that have none of it: kUnpad operations whose destinations are device-visible
// addresses of pinned host memory.  Returns false, and takes nothing, where that launch has no workgroups to spare.
bool core_copy_beside(flstm_core_plan* plan, bool forward, const OpList& copies);

}  // namespace flstm_hip
