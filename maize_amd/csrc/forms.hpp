// The launcher's own forms: kernels it runs in place of the registry kernel that select_kernel names, when the caller names
// none and the cost model has them faster.  Host logic only; no HIP calls.
//
// They are to the registry what the tail split is: the same product, composed differently.  maize_hip_gemm_plan and
// maize_hip_gemm_select keep reporting the registry kernel, whose requirements and arithmetic (8-bit operands: multiplied as
// they are, or widened) the form shares; maize_hip_gemm_ex_form reports the form.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include "maize_hip.h"

namespace maize {

constexpr uint32_t kMaxForms = 80;
uint32_t form_count();
const char* form_name(uint32_t index);     // kernel of the tile code object; NULL: an unused index

struct FormPlan {
    uint32_t kernel;           // form index
    uint32_t grid, ksplit;     // grid.x of 256-thread workgroups; K ranges per tile
    size_t workspace_bytes;    // 0, or ticket counters and the ranges' partial tiles
};
// Whether one of the forms is to run `d` instead of registry kernel `registry` (its index), and how.
bool choose_form(const maize_gemm_ex_desc_t& d, uint32_t registry, uint32_t compute_units, FormPlan* out);

}  // namespace maize
