// Routing of dense Boolean steps to the int8 MFMA kernel (dense.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/tensorsat_amd.h"

namespace tsd {

// True when the step is a K-innermost two-operand product with at least 2^6 contracted
// entries and at least 4 lhs-only and 4 rhs-only out bits, operands 16-byte aligned, and
// the MFMA route is enabled (ts_dense_config).
bool dense_eligible(const ts_step& st, const void* lhs, const void* rhs);

constexpr int DENSE_GANG = 64;  // jobs of one launch

// True when two records differ at most in their operands' offsets.
bool same_dense_step(const ts_step& x, const ts_step& y);

// The step on n (1..DENSE_GANG) sets of operands in one launch.
int launch_dense(int n, const uint8_t* const* lhs, const uint8_t* const* rhs, uint8_t* const* out, const ts_step& st,
                 int mode, hipStream_t s);

}  // namespace tsd
