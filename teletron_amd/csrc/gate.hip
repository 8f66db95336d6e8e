// Instantiates the gated-residual kernel family (forward and backward).
#include "kernel_table.hpp"

namespace tt {
KernelInfo gate_fwd_kernel(bool narrow, int idx, int rows) { return lookup_gate<kGateFwd>(narrow, idx, rows); }
KernelInfo gate_bwd_kernel(bool narrow, int idx, int rows) { return lookup_gate<kGateBwd>(narrow, idx, rows); }
}  // namespace tt
