// The kept entries of softmax rows wait in a slab (one word each: column low, bf16 bits high; `cap` words a row) until the CSR offsets
// are known (softmax.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hyc {

// rows with at most `cap` entries from the slab to the CSR arrays; rows with more are left to the caller
void launch_slab_copy(int64_t rows, const int32_t* counts, const uint32_t* slab, int64_t cap, const int32_t* row_ptr, int32_t* cols, void* vals,
                      hipStream_t stream);

}  // namespace hyc
