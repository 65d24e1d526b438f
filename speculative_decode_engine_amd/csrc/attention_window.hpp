// Causal paged GQA attention for wide windows (prompts and prompt chunks):
// attention_window.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "sde/attention_device.hpp"

namespace sde {
namespace win {

constexpr int kWinWaves = 8;                // waves per workgroup: 4 row blocks x 2 token halves
constexpr int kWinRows = 32 * 4;            // (query, head in group) rows per workgroup
constexpr int kWinTok = 64;                 // tokens per tile

struct WindowPlan {
  int row_groups;      // ceil(R / kWinRows)
  int n_parts;         // context partitions of a row group
  int tiles_per_part;  // tiles of kWinTok tokens per partition
};

// Whether a window of R rows per KV head over L_max keys runs here instead
// of on the 16-row tile kernels (head sizes 64 / 128, block sizes those
// kernels take).
bool window_serves(int L_max, int nkv, int R);

// The plan of such a window; partials never exceed `max_bytes` and never
// `max_parts` partitions.
WindowPlan window_plan(int L_max, int nkv, int R, int dph, int n_cus, int max_parts,
                       size_t max_bytes);

size_t window_partial_bytes(const WindowPlan& p, int nkv, int R, int dph);

// Launches it (dph 64 or 128): a.src, q, out, partials, nh, nkv, G, R,
// pos_base and qscale are read, the rest is the plan's.
int window_attention(const attn::AttnArgs& a, const WindowPlan& p, int dph, hipStream_t stream);

}  // namespace win
}  // namespace sde
