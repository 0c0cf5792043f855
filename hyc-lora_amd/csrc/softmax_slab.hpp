// The kept entries of softmax rows wait in a slab (one word each: column low, bf16 bits high; `cap` words a row) until the CSR offsets
// are known (softmax.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hyc {

// rows with at most `cap` entries from the slab to the CSR arrays; rows with more are left to the caller
void launch_slab_copy(int64_t rows, const int32_t* counts, const uint32_t* slab, int64_t cap, const int32_t* row_ptr, int32_t* cols, void* vals,
                      hipStream_t stream);

// Offsets and copy in one launch, up to this many rows: a workgroup of 256 threads takes four rows and adds up the counts in front of them
// itself, 4 bytes a row from L2, so what the launch reads grows with the square of the rows.  Two launches -> one, softmax rows with
// 1 % of 2048 entries kept, us: up to 1024 rows 9.0 -> 2.7, 2048 9.2 -> 3.1, 4096 9.2 -> 3.7, 6000 5.9 -> 4.1, 8192 6.1 -> 5.2.
constexpr int64_t SLAB_OFFSETS_MAX = 8192;

struct RowRoom { int64_t base; int limit, n; };            // first entry, room and number of entries of a wave's row
// the wave's row is 4 blockIdx.x + wave; every thread takes part; counts 16-byte aligned; row_ptr and *total (may be null) as hyc_csr_offsets
// leaves them
__device__ __forceinline__ RowRoom csr_rows4(const int32_t* __restrict__ counts, int64_t rows, int64_t capacity, int32_t* __restrict__ row_ptr,
                                             int64_t* __restrict__ total) {
  __shared__ long long part[4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int64_t r0 = (int64_t)blockIdx.x * 4, row = r0 + wave;
  long long sum = 0;
#pragma unroll 4
  for (int64_t i = 4 * (int64_t)threadIdx.x; i < r0; i += 1024) {      // (r0 is a multiple of 4)
    const int4 v = *reinterpret_cast<const int4*>(counts + i);
    sum += ((long long)v.x + v.y) + ((long long)v.z + v.w);
  }
#pragma unroll
  for (int d = 32; d; d >>= 1) sum += __shfl_xor(sum, d, 64);
  if (lane == 0) part[wave] = sum;
  __syncthreads();
  long long at = (part[0] + part[1]) + (part[2] + part[3]);
  int n = 0;
  for (int k = 0; k <= wave; ++k) {
    at += n;
    n = r0 + k < rows ? counts[r0 + k] : 0;
  }
  const long long end = at + n, from = at < capacity ? at : capacity, to = end < capacity ? end : capacity;
  if (lane == 0 && row < rows) {
    row_ptr[row] = (int32_t)from;
    if (row + 1 == rows) {
      row_ptr[rows] = (int32_t)to;
      if (total) *total = end;
    }
  }
  return {from, (int)(to - from), n};
}

}  // namespace hyc
