// What the attention kernels (attn.hip, attn_kept.hip) share: operand views, LDS tiles of walked rows and their swizzle, MFMA
// fragments, the write-out of owned rows, which block a workgroup takes, and the checks of the entry points.
#pragma once
#include <math.h>

#include "abi_util.hpp"
#include "row_kernels.hpp"

namespace hyc {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

constexpr int AT_OWN = 128;      // rows a workgroup owns (four waves of 32)
constexpr int AT_WALK = 64;      // rows of a walked tile
constexpr float LOG2E = 1.44269504088896340736f, LN2 = 0.693147180559945309417f;

// one [B, S, heads, hd] operand: token s of batch element b and head h starts at p + (b S + s) pitch + h hd
struct AttnRows {
  const uint16_t* p;
  int64_t pitch;
};
struct AttnOut {
  uint16_t* p;
  int64_t pitch;
};

// chunk position swizzle of an LDS tile with HD / 8 chunks per row.  Reading one chunk column of 16 consecutive rows and
// the 4 x 4 chunks a transposing read touches (rows r .. r+7, four neighbouring chunks) must both spread over the banks:
// a 256-byte span holds one row of 16 chunks or two rows of 8.
template <int HD>
__device__ __forceinline__ int swz(int row) {
  if (HD == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
  return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}

__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// every load to LDS of this wave has landed, then the workgroup meets
__device__ __forceinline__ void tile_barrier() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// One matrix of a walked tile: rows [row0, row0 + ROWS) of `rsrc` (rows past the last one repeat it: finite values whose
// weight is zero) to the LDS tile at `lds`.
template <int HD, int ROWS = AT_WALK>
__device__ __forceinline__ void issue_tile(u32x4_t rsrc, uint32_t pitch_bytes, int row0, int last_row, uint32_t lds) {
  constexpr int CH = HD / 8, RPI = 64 / CH;                 // chunks per row, rows per instruction
  constexpr int N = ROWS / (4 * RPI);                     // instructions per wave
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int r = (wave + 4 * u) * RPI + lane / CH;
    const int c = (lane % CH) ^ swz<HD>(r);
    const int row = row0 + r < last_row ? row0 + r : last_row;
    dma_b128(rsrc, (uint32_t)row * pitch_bytes + 16u * (uint32_t)c, lds + (uint32_t)(wave + 4 * u) * 1024u);
  }
}

// A lane's LDS addresses within a tile (bytes), from which every fragment address is one exclusive-or and an immediate:
// tiles start at multiples of 1024 and the chunk number lies in address bits 4 to 6 (7), which the row number leaves alone.
template <int HD>
struct TileLane {
  uint32_t rows, cols;
  __device__ __forceinline__ void init(uint32_t tile) {
    const int lane = threadIdx.x & 63, r = lane & 31, g = lane >> 4, s = lane & 15;
    rows = tile + (uint32_t)(r * HD * 2 + (((lane >> 5) ^ swz<HD>(r)) << 4));
    const int rr = 4 * (g >> 1) + (s >> 2), col = 16 * (g & 1) + 4 * (s & 3);
    cols = tile + (uint32_t)(rr * HD * 2 + (((col >> 3) ^ swz<HD>(rr)) << 4) + (col & 7) * 2);
  }
  // the same lane in another tile.  Opaque to the compiler, which would otherwise keep all 2 * 16 derived addresses of every
  // tile in registers across the loop (and spill operands for them).
  __device__ __forceinline__ TileLane in(uint32_t offset) const {
    TileLane t = {rows + offset, cols + offset};
    asm volatile("" : "+v"(t.rows), "+v"(t.cols));
    return t;
  }
};
typedef const bf16x8_t __attribute__((address_space(3))) * lds_b128;
typedef bf16x4_t __attribute__((address_space(3))) * lds_b64;
// operand fragment, rows from the tile as stored: lane l gets the 8 elements [16 ks + 8 (l / 32), +8) of row row0 + l % 32
// of the matrix `mat` bytes behind the lane's tile
template <int HD>
__device__ __forceinline__ bf16x8_t frag_rows(const TileLane<HD>& t, uint32_t mat, int row0, int ks) {
  return *(lds_b128)(uintptr_t)((t.rows ^ (uint32_t)(ks << 5)) + mat + (uint32_t)(row0 * HD * 2));
}
// operand fragment, columns of the tile as operand rows: lane l gets column col0 + l % 32 of the 8 rows
// {0-3, 8-11} (l < 32) or {4-7, 12-15} (l >= 32) of the 16 starting at row0 (a multiple of 16; swz(r + 8) = swz(r) ^ 2)
template <int HD>
__device__ __forceinline__ bf16x8_t frag_cols(const TileLane<HD>& t, uint32_t mat, int col0, int row0) {
  const uint32_t x = (uint32_t)(col0 << 1), off = mat + (uint32_t)(row0 * HD * 2);
  const bf16x4_t a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_b64)(uintptr_t)((t.cols ^ x) + off));
  const bf16x4_t b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_b64)(uintptr_t)((t.cols ^ x ^ 32u) + off + (uint32_t)(8 * HD * 2)));
  bf16x8_t f;
  f[0] = a[0]; f[1] = a[1]; f[2] = a[2]; f[3] = a[3];
  f[4] = b[0]; f[5] = b[1]; f[6] = b[2]; f[7] = b[3];
  return f;
}
// the wave's own 32 rows as operand fragments, from memory (rows past the last one repeat it)
template <int HD>
__device__ __forceinline__ void load_own(const uint16_t* base, uint32_t pitch_bytes, int row0, int last_row, bf16x8_t (&f)[HD / 16]) {
  const int lane = threadIdx.x & 63;
  const int row = row0 + (lane & 31) < last_row ? row0 + (lane & 31) : last_row;
  const char* p = reinterpret_cast<const char*>(base) + (uint64_t)((uint32_t)row * pitch_bytes + 16u * (lane >> 5));
#pragma unroll
  for (int ks = 0; ks < HD / 16; ++ks) {
    const uint4 v = *reinterpret_cast<const uint4*>(p + 32 * ks);
    f[ks] = __builtin_bit_cast(bf16x8_t, v);
  }
}
// the eight values [8 half, 8 half + 8) of an accumulator as a bf16 operand fragment
__device__ __forceinline__ bf16x8_t acc_frag(const floatx16_t& a, int half) {
  uint4 v;
  v.x = pack_bf16(a[8 * half + 0], a[8 * half + 1]);
  v.y = pack_bf16(a[8 * half + 2], a[8 * half + 3]);
  v.z = pack_bf16(a[8 * half + 4], a[8 * half + 5]);
  v.w = pack_bf16(a[8 * half + 6], a[8 * half + 7]);
  return __builtin_bit_cast(bf16x8_t, v);
}
__device__ __forceinline__ floatx16_t zero16() {
  floatx16_t z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}
__device__ __forceinline__ float other_half(float v) { return __shfl_xor(v, 32, 64); }
#define HYC_MFMA(a_, b_, c_) __builtin_amdgcn_mfma_f32_32x32x16_bf16(a_, b_, c_, 0, 0, 0)

// Write a wave's result, held transposed (o[db][i] = row l % 32, column 32 db + 8 (i / 4) + 4 (l / 32) + i % 4), as bf16 rows
// of `out`: through 32 * HD elements of LDS of the wave's own, so that a row leaves as whole 16-byte chunks.
// cosv: undo the rotary embedding on the way (rows are positions row0 + r): gradients of rotated q / k.
template <int HD>
__device__ __forceinline__ void store_own(floatx16_t (&o)[HD / 32], uint16_t* T, uint16_t* out, int64_t pitch, int row0, int rows,
                                          const uint16_t* cosv, const uint16_t* sinv) {
  constexpr int NB = HD / 32, CH = HD / 8;
  const int lane = threadIdx.x & 63, r = lane & 31, hi = lane >> 5;
  if (cosv) {
    const int pos = row0 + r < rows ? row0 + r : rows - 1;
#pragma unroll
    for (int db = 0; db < NB / 2; ++db)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int64_t at = (int64_t)pos * HD + 32 * db + 8 * b + 4 * hi;
        const uint2 cl = *reinterpret_cast<const uint2*>(cosv + at), sl = *reinterpret_cast<const uint2*>(sinv + at);
        const uint2 ch = *reinterpret_cast<const uint2*>(cosv + at + HD / 2), sh = *reinterpret_cast<const uint2*>(sinv + at + HD / 2);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint32_t c0 = t < 2 ? cl.x : cl.y, s0 = t < 2 ? sl.x : sl.y, c1 = t < 2 ? ch.x : ch.y, s1 = t < 2 ? sh.x : sh.y;
          const float fcl = (t & 1) ? bf_hi(c0) : bf_lo(c0), fsl = (t & 1) ? bf_hi(s0) : bf_lo(s0);
          const float fch = (t & 1) ? bf_hi(c1) : bf_lo(c1), fsh = (t & 1) ? bf_hi(s1) : bf_lo(s1);
          const float lo = o[db][4 * b + t], hh = o[db + NB / 2][4 * b + t];
          o[db][4 * b + t] = __builtin_fmaf(lo, fcl, hh * fsh);
          o[db + NB / 2][4 * b + t] = __builtin_fmaf(hh, fch, -(lo * fsl));
        }
      }
  }
#pragma unroll
  for (int db = 0; db < NB; ++db)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int c = 4 * db + b;
      const uint2 w = make_uint2(pack_bf16(o[db][4 * b], o[db][4 * b + 1]), pack_bf16(o[db][4 * b + 2], o[db][4 * b + 3]));
      *reinterpret_cast<uint2*>(T + r * HD + 8 * (c ^ swz<HD>(r)) + 4 * hi) = w;
    }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the other lanes' writes before these reads
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int u = 0; u < 32 * CH / 64; ++u) {
    const int at = lane + 64 * u, rr = at / CH, c = at % CH;
    if (row0 + rr < rows)
      *reinterpret_cast<uint4*>(out + (int64_t)(row0 + rr) * pitch + 8 * c) =
          *reinterpret_cast<const uint4*>(T + rr * HD + 8 * (c ^ swz<HD>(rr)));
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // and the reads before what is written there next
  __builtin_amdgcn_wave_barrier();
}

// Which block of owned rows and which head a workgroup takes.  Workgroups of one head come BH apart, so with a multiple
// of 8 heads they share an XCD and its L2.  The blocks with the longest walk go first; when the whole launch is resident
// at once (two workgroups per CU) the second half runs from the shortest up, so that a CU gets a long and a short one.
__device__ __forceinline__ void attn_block(int blocks, int BH, bool long_is_last, int* block, int* bh) {
  const int L = blockIdx.x, r = L / BH;
  *bh = L - r * BH;
  int rank = r;                                             // 0 = longest walk
  if (blocks * BH <= 512) {
    const int first = (blocks + 1) / 2;
    rank = r < first ? r : blocks - 1 - (r - first);
  }
  *block = long_is_last ? blocks - 1 - rank : rank;
}
inline int attn_args(const char* who, int64_t B, int64_t S, int64_t heads, int64_t hd, float scale, const int64_t* pitches, int n) {
  if (B < 0 || S < 0 || heads <= 0) return fail(HYC_EINVAL, "%s: B=%lld S=%lld heads=%lld", who, (long long)B, (long long)S, (long long)heads);
  if (hd != 64 && hd != 128) return fail(HYC_ENOTSUP, "%s: head_dim=%lld (64 or 128)", who, (long long)hd);
  // (the running maximum and the mask are taken before the scores are scaled, and the backward divides by the scale)
  if (!(scale > 0.f) || !(1.0f / scale > 0.f) || !isfinite(1.0f / scale))
    return fail(HYC_EINVAL, "%s: scale=%g must be positive, and so must its reciprocal, both finite", who, (double)scale);
  for (int i = 0; i < n; ++i) {
    if (pitches[i] < heads * hd || pitches[i] % 8 != 0)
      return fail(HYC_EINVAL, "%s: token pitch %lld (at least heads*head_dim, a multiple of 8)", who, (long long)pitches[i]);
    if (S * pitches[i] >= ((int64_t)1 << 30))
      return fail(HYC_ENOTSUP, "%s: S * pitch = %lld elements (a batch element must stay below 2 GiB)", who, (long long)(S * pitches[i]));
  }
  const int64_t blocks = (S + AT_OWN - 1) / AT_OWN;
  if (B * heads * blocks >= ((int64_t)1 << 24))          // (a launch counts its threads in 32 bits)
    return fail(HYC_ENOTSUP, "%s: B * heads * S = %lld matrices of %lld blocks", who, (long long)(B * heads), (long long)blocks);
  return HYC_OK;
}

}  // namespace hyc
