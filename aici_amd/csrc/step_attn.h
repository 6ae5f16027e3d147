// The attention of a step with both prompt chunks and decode rows in one launch.
#pragma once

#include "paged_decode.h"
#include "prefill_common.h"

namespace hipattn {

// `rows` null: chunks alone, whose keys are dealt out to more workgroups.  Enqueues it, or returns false, having enqueued nothing, where the two have to go by themselves (other head sizes, types or block sizes, a
// capture, shapes that are faster so).  Throws what the two entry points' own checks would.
bool step_attention(const PagedPrefillCall &chunks, hipattn_tensor *chunks_out, const DecodeCall *rows, hipattn_tensor *rows_out, void *stream);

}  // namespace hipattn
