// stablehlo.sort / chlo.top_k library steps.
#pragma once

#include <vector>

#include "ir.h"
#include "runtime.h"

namespace pjrtx {

// Fails with UNIMPLEMENTED / INVALID_ARGUMENT when the op (its comparator,
// operand count, key type or k) is outside what run_sort handles.
void check_sort_supported(const Program& prog, const Op& op);

// Bytes of device scratch the op takes where `max_bytes` are to be had.
int64_t sort_op_scratch(const Program& prog, const Op& op, int64_t max_bytes);

// Writes the op's results (allocated by the caller) on the device's stream.
void run_sort(Device* dev, const Program& prog, const Op& op, std::vector<MemRef>& vals);

}  // namespace pjrtx
