// The experts' products in large tiles (moe_tiled.hip), as moe.hip launches them.
#pragma once

#include "common.h"
#include "microllm_hip.h"

namespace mll {

// FORM of moe_grouped_kernel by number; the pairs are sorted (offsets, order). k is a multiple of 64 and n_out of 8, `a`, `w` and `x` begin at
// 16-byte boundaries, and the rows of `a` and an expert's weight take less than 4 GB each.
int launch_moe_tiled(int form_number, const bf16* a, const bf16* w, const int32_t* offsets, const int32_t* order, const float* weights, int n_out,
                     int k, void* out, int top, int n_tokens, int weight_on_input, int from_tokens, const bf16* x, const MllExpertForm& form,
                     hipStream_t stream);

}  // namespace mll
