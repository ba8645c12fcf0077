#pragma once
#include "attn_common.h"
namespace spx {
// The launch of attn.hip's exact / exact + tail attention (bf16 output) with one query
// tile per workgroup; no work queue.
void launch_attn_solo(const AttnArgs& a, bool tail, hipStream_t st);
}  // namespace spx
