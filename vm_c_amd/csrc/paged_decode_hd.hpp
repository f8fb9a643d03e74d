// paged_decode_hd.hpp -- the MFMA page decode of head_dim 64 and 256, for the
// entry points in paged_decode.hip.
#pragma once

#include "generic_attn.hpp"

namespace vmc {

// whether paged_decode_hd takes this call of gen_attention (checked operands)
bool paged_decode_hd_takes(const GenArgs& a);
// The same rows as gen_attention(a).  ws / ws_bytes: fp32 partial rows of
// sequences cut over page ranges (may be null: no row is cut); max_splits as
// vmc_paged_attention_decode's.
int paged_decode_hd(const GenArgs& a, int max_splits, void* ws, size_t ws_bytes, hipStream_t stream);

}  // namespace vmc
