// The threshold scheme's kernels for the common row shapes (threshold.hip), as compress.hip reaches them.
#pragma once
#include "abi_util.hpp"

namespace hyc {

// x_hat of codes + CSR outliers; false (nothing launched) for rows these kernels do not cover
bool launch_thr_restore(const void* stored, int64_t M, int64_t H, const RowGeom& g, const ThrArgs& a, bool perchan, void* xhat, hipStream_t stream);

}  // namespace hyc
