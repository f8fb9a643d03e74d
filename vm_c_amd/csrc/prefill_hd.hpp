// prefill_hd.hpp -- the MFMA prefill of head_dim 64 and 256 over this step's
// K/V rows, for the entry points in prefill.hip.
#pragma once

#include "generic_attn.hpp"

namespace vmc {

// whether prefill_hd takes this call of gen_attention (checked operands)
bool prefill_hd_takes(const GenArgs& a);
// the same rows as gen_attention(a)
int prefill_hd(const GenArgs& a, hipStream_t stream);

}  // namespace vmc
