// Prefill launches whose keys are shared out over workgroups (prefill.hip).
#pragma once

#include "tla_internal.h"

namespace tla {

// Where several workgroups share a query tile, each leaves its waves' softmax
// states here and the last to arrive merges them.  One fixed size for every
// shape (a shape that needs more is not shared out), so the workspace is
// allocated once, by the first launch that shares one, and no later launch
// replaces it.
constexpr int kPrefillStateBytes = 34 * 64 * 4;
constexpr int kPrefillStates = 6144;
constexpr int kPrefillCounters = 4096;  // arrivals, zero between launches

// Whether launch_prefill_short (append and attention in one launch) is the
// faster way for this shape.
bool prefill_is_short(int n_lb, int n_head_kv, int gqa, int pos0, int n_tok);
// Whether that launch (short_launch) or launch_prefill_attention has several
// workgroups to a query tile: only then part and counters are used.
bool prefill_shares(bool short_launch, int n_lb, int n_head_kv, int gqa, int pos0, int n_tok);
// p.kvp and p.n_ptiles are not used.
hipError_t launch_prefill_short(const PrefillParams& p, float* part, int* counters, hipStream_t s);

// Attention over the planes that launch_prefill_append wrote.
hipError_t launch_prefill_attention(const PrefillParams& p, float* part, int* counters, hipStream_t s);

}  // namespace tla
