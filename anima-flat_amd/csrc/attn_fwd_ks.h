// The key-split forward for short query ranges (attn_fwd_ks.hip).
#pragma once

#include "attn_fwd.h"

namespace aa {

constexpr int kKsQueries = 64;  // queries per workgroup

// Launches the key-split kernel over the B H ceil(Sq / 64) workgroups of p's
// problem (B = batch size). Writes O (and LSE) in one pass, with no workspace.
void launch_attn_fwd_ks(const FwdParams& p, int64_t B, hipStream_t stream);

}  // namespace aa
