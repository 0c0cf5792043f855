// Causal attention on the [B, S, heads * hd] rows the projections produce (q and k after RoPE), forward and backward,
// without an [S, S] matrix and without a head-major copy of anything.  (The reference reaches its fused attention through
// flash_attn, operators/efficient_flashattention.py:10-135.)
//
//   forward    O = softmax(scale Q K^T + causal) V,  lse[q] = log sum_k exp(scale q.k)
//   backward   P = exp(scale Q K^T - lse),  dV = P^T dO,  dS = P o (dO V^T - delta),  dQ = scale dS K,  dK = scale dS^T Q
//              with delta[q] = sum_d dO[q, d] O[q, d]
//
// What bounds these kernels is that a wave's steps follow each other: scores, exponentials, second product.  No unit is full; as
// shares of the kernel's cycles at 4 x 1024 x 32 heads x 128 (55, 66 and 87 us; counters): matrix cores 0.34 forward, 0.44 dQ,
// 0.42 dK / dV; the other vector instructions 0.40, 0.24 and 0.21, the exponentials' slower rate not counted (about 0.1
// more); LDS 0.20, 0.25 and 0.30, of which 7 % at most bank conflicts.  The registers leave room for two waves per SIMD to
// overlap them, so everything that can stay in registers does, and every fragment is read as few times as it can be:
//  * A wave owns 32 queries (forward, dQ) or 32 keys (dK / dV) and keeps their rows as MFMA operands for the whole loop.
//  * The score tile is produced with the owned index in the lane (column) and the walked index in the registers (row), so
//    softmax statistics are one value per lane, and the 16 scores of a lane, rounded to bf16, ARE the operand of the second
//    product: its reduction runs over the walked index in the order {0-3, 8-11 | 4-7, 12-15} the accumulator layout gives,
//    and the other operand is fetched from LDS in the same order by the transposing read (ds_read_b64_tr_b16).
//  * The walked tiles (64 rows of two matrices, 32 KB) go from memory straight to LDS, double-buffered, one barrier per
//    tile; two workgroups of four waves share a CU.
//  * Rows are 16-byte chunks stored at chunk ^ f(row), which makes both the row-wise 16-byte reads and the transposing
//    reads use all 64 banks evenly without padding (the direct load to LDS cannot pad).
// dQ and dK / dV are two kernels (7 products instead of 5): no atomics, the results do not depend on arrival order.
// At head_dim 128 dK / dV takes all 256 registers and keeps five values that do not change in the loop in scratch, dQ one (5 and 1
// MB written once, in front of the loop, by the counters of memory traffic).
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

// One matrix of a walked tile: rows [row0, row0 + 64) of `rsrc` (rows past the last one repeat it: finite values whose
// weight is zero) to the LDS tile at `lds`.
template <int HD>
__device__ __forceinline__ void issue_tile(u32x4_t rsrc, uint32_t pitch_bytes, int row0, int last_row, uint32_t lds) {
  constexpr int CH = HD / 8, RPI = 64 / CH;                 // chunks per row, rows per instruction
  constexpr int N = AT_WALK / (4 * RPI);                    // instructions per wave
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

template <int HD>
__global__ void __launch_bounds__(256, 2)
k_attn_fwd(AttnRows Q, AttnRows K, AttnRows V, AttnOut O, float* __restrict__ lse, int S, int heads, int BH, int blocks, float scale) {
  constexpr int KS = HD / 16, NB = HD / 32;
  __shared__ __align__(1024) uint16_t lds[4 * AT_WALK * HD];            // [buffer][K, V] tiles
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hi = lane >> 5;
  int block, bh;
  attn_block(blocks, BH, true, &block, &bh);
  const int b = bh / heads, h = bh - b * heads;
  const int q0 = block * AT_OWN, w0 = q0 + 32 * wave;
  auto rows_of = [&](const AttnRows& t) { return t.p + (int64_t)b * S * t.pitch + (int64_t)h * HD; };
  auto bytes_of = [&](const AttnRows& t) { return (uint32_t)(((int64_t)(S - 1) * t.pitch + HD) * 2); };
  const u32x4_t rk = uniform_rsrc(rows_of(K), bytes_of(K)), rv = uniform_rsrc(rows_of(V), bytes_of(V));
  const uint32_t pk = (uint32_t)K.pitch * 2u, pv = (uint32_t)V.pitch * 2u;
  const uint32_t base = lds_offset(lds);
  constexpr uint32_t TB = AT_WALK * HD * 2;                             // bytes of a tile
  TileLane<HD> lane_at;
  lane_at.init(base);
  const int q_end = q0 + AT_OWN < S ? q0 + AT_OWN : S;
  const int tiles = (q_end + AT_WALK - 1) / AT_WALK;
  issue_tile<HD>(rk, pk, 0, S - 1, base);
  issue_tile<HD>(rv, pv, 0, S - 1, base + TB);
  bf16x8_t qf[KS];
  load_own<HD>(rows_of(Q), (uint32_t)Q.pitch * 2u, w0, S - 1, qf);
  floatx16_t o[NB];
#pragma unroll
  for (int d = 0; d < NB; ++d) o[d] = zero16();
  const float c = scale * LOG2E;
  // the running maximum starts below every score but finite, also once scaled: a row that has met only scores of -inf so far
  // (masked keys, products past the range) keeps it, and weights them 0
  float m = -3e38f / __builtin_fmaxf(c, 1.f), l = 0.f;
  const int my_q = w0 + (lane & 31);
  for (int t = 0; t < tiles; ++t) {
    tile_barrier();
    if (t + 1 < tiles) {
      issue_tile<HD>(rk, pk, (t + 1) * AT_WALK, S - 1, base + ((t + 1) & 1) * 2 * TB);
      issue_tile<HD>(rv, pv, (t + 1) * AT_WALK, S - 1, base + ((t + 1) & 1) * 2 * TB + TB);
    }
    const int k0 = t * AT_WALK;
    if (k0 > w0 + 31) continue;                                         // (the same for the whole wave) all of it above the diagonal
    const TileLane<HD> T = lane_at.in((t & 1) * 2 * TB);                // K; V is TB bytes behind
    floatx16_t s[2] = {zero16(), zero16()};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) s[kb] = HYC_MFMA(frag_rows<HD>(T, 0, 32 * kb, ks), qf[ks], s[kb]);
    if (k0 + AT_WALK - 1 > w0) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (k0 + 32 * kb + 8 * (i >> 2) + 4 * hi + (i & 3) > my_q) s[kb][i] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = __builtin_fmaxf(mx, s[kb][i]);
    mx = __builtin_fmaxf(mx, other_half(mx));
    if (__ballot(mx > m)) {
      // (mx is -inf where a row of the wave lies wholly above this tile: m keeps its value)
      const float mn = __builtin_fmaxf(m, mx), f = __builtin_amdgcn_exp2f((m - mn) * c);
      m = mn;
      l *= f;
#pragma unroll
      for (int d = 0; d < NB; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] *= f;
    }
    const float mc = m * c;
    float sum = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[kb][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][i], c, -mc));
        sum += s[kb][i];
      }
    l += sum;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const bf16x8_t pf = acc_frag(s[ks >> 1], ks & 1);
#pragma unroll
      for (int d = 0; d < NB; ++d) o[d] = HYC_MFMA(frag_cols<HD>(T, TB, 32 * d, 16 * ks), pf, o[d]);
    }
  }
  l += other_half(l);
  const float inv = 1.0f / l;
#pragma unroll
  for (int d = 0; d < NB; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] *= inv;
  if (hi == 0 && my_q < S) lse[(int64_t)bh * S + my_q] = (m * c + __builtin_amdgcn_logf(l)) * LN2;
  __syncthreads();                                                      // the tiles are no longer read
  store_own<HD>(o, lds + wave * 32 * HD, O.p + (int64_t)b * S * O.pitch + (int64_t)h * HD, O.pitch, w0, S, nullptr, nullptr);
}

// dQ: owns queries, walks keys.
template <int HD>
__global__ void __launch_bounds__(256, 2)
k_attn_bwd_dq(AttnRows Q, AttnRows K, AttnRows V, AttnRows G, const float* __restrict__ nlse, const float* __restrict__ ndelta,
              const uint16_t* __restrict__ cosv, const uint16_t* __restrict__ sinv, AttnOut DQ, int S, int heads, int BH, int blocks, float scale) {
  constexpr int KS = HD / 16, NB = HD / 32;
  __shared__ __align__(1024) uint16_t lds[4 * AT_WALK * HD];            // [buffer][K, V] tiles
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hi = lane >> 5;
  int block, bh;
  attn_block(blocks, BH, true, &block, &bh);
  const int b = bh / heads, h = bh - b * heads;
  const int q0 = block * AT_OWN, w0 = q0 + 32 * wave;
  auto rows_of = [&](const AttnRows& t) { return t.p + (int64_t)b * S * t.pitch + (int64_t)h * HD; };
  auto bytes_of = [&](const AttnRows& t) { return (uint32_t)(((int64_t)(S - 1) * t.pitch + HD) * 2); };
  const u32x4_t rk = uniform_rsrc(rows_of(K), bytes_of(K)), rv = uniform_rsrc(rows_of(V), bytes_of(V));
  const uint32_t pk = (uint32_t)K.pitch * 2u, pv = (uint32_t)V.pitch * 2u;
  const uint32_t base = lds_offset(lds);
  constexpr uint32_t TB = AT_WALK * HD * 2;
  TileLane<HD> lane_at;
  lane_at.init(base);
  const int q_end = q0 + AT_OWN < S ? q0 + AT_OWN : S;
  const int tiles = (q_end + AT_WALK - 1) / AT_WALK;
  issue_tile<HD>(rk, pk, 0, S - 1, base);
  issue_tile<HD>(rv, pv, 0, S - 1, base + TB);
  bf16x8_t qf[KS], gf[KS];
  load_own<HD>(rows_of(Q), (uint32_t)Q.pitch * 2u, w0, S - 1, qf);
  load_own<HD>(rows_of(G), (uint32_t)G.pitch * 2u, w0, S - 1, gf);
  const int my_q = w0 + (lane & 31), at_q = my_q < S ? my_q : S - 1;
  const float c = scale * LOG2E, ml = nlse[(int64_t)bh * S + at_q], md = ndelta[(int64_t)bh * S + at_q];
  floatx16_t o[NB];
#pragma unroll
  for (int d = 0; d < NB; ++d) o[d] = zero16();
  for (int t = 0; t < tiles; ++t) {
    tile_barrier();
    if (t + 1 < tiles) {
      issue_tile<HD>(rk, pk, (t + 1) * AT_WALK, S - 1, base + ((t + 1) & 1) * 2 * TB);
      issue_tile<HD>(rv, pv, (t + 1) * AT_WALK, S - 1, base + ((t + 1) & 1) * 2 * TB + TB);
    }
    const int k0 = t * AT_WALK;
    if (k0 > w0 + 31) continue;
    const TileLane<HD> T = lane_at.in((t & 1) * 2 * TB);                // K; V is TB bytes behind
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      floatx16_t s, dp;                                                 // the accumulators start at -lse / scale and -delta
#pragma unroll
      for (int i = 0; i < 16; ++i) { s[i] = ml; dp[i] = md; }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        s = HYC_MFMA(frag_rows<HD>(T, 0, 32 * kb, ks), qf[ks], s);
        dp = HYC_MFMA(frag_rows<HD>(T, TB, 32 * kb, ks), gf[ks], dp);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(s[i] * c) * dp[i];
      if (k0 + 32 * kb + 31 > w0) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (k0 + 32 * kb + 8 * (i >> 2) + 4 * hi + (i & 3) > my_q) s[i] = 0.f;
      }
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const bf16x8_t df = acc_frag(s, half);
#pragma unroll
        for (int d = 0; d < NB; ++d) o[d] = HYC_MFMA(frag_cols<HD>(T, 0, 32 * d, 32 * kb + 16 * half), df, o[d]);
      }
    }
  }
#pragma unroll
  for (int d = 0; d < NB; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] *= scale;
  __syncthreads();
  store_own<HD>(o, lds + wave * 32 * HD, DQ.p + (int64_t)b * S * DQ.pitch + (int64_t)h * HD, DQ.pitch, w0, S, cosv, sinv);
}

// dK and dV: owns keys, walks queries from the diagonal on.
template <int HD>
__global__ void __launch_bounds__(256, 2)
k_attn_bwd_dkdv(AttnRows Q, AttnRows K, AttnRows V, AttnRows G, const float* __restrict__ nlse, const float* __restrict__ ndelta,
                const uint16_t* __restrict__ cosv, const uint16_t* __restrict__ sinv, AttnOut DK, AttnOut DV, int S, int heads, int BH,
                int blocks, float scale) {
  constexpr int KS = HD / 16, NB = HD / 32;
  __shared__ __align__(1024) uint16_t lds[4 * AT_WALK * HD];            // [buffer][Q, dO] tiles
  __shared__ __align__(256) float stats[4 * AT_WALK];                   // [buffer][-lse / scale, -delta]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hi = lane >> 5;
  int block, bh;
  attn_block(blocks, BH, false, &block, &bh);
  const int b = bh / heads, h = bh - b * heads;
  const int k0 = block * AT_OWN, w0 = k0 + 32 * wave;
  auto rows_of = [&](const AttnRows& t) { return t.p + (int64_t)b * S * t.pitch + (int64_t)h * HD; };
  auto bytes_of = [&](const AttnRows& t) { return (uint32_t)(((int64_t)(S - 1) * t.pitch + HD) * 2); };
  const u32x4_t rq = uniform_rsrc(rows_of(Q), bytes_of(Q)), rg = uniform_rsrc(rows_of(G), bytes_of(G));
  const u32x4_t rl = uniform_rsrc(nlse + (int64_t)bh * S, (uint32_t)S * 4u), rd = uniform_rsrc(ndelta + (int64_t)bh * S, (uint32_t)S * 4u);
  const uint32_t pq = (uint32_t)Q.pitch * 2u, pg = (uint32_t)G.pitch * 2u;
  const uint32_t base = lds_offset(lds), sbase = lds_offset(stats);
  constexpr uint32_t TB = AT_WALK * HD * 2;
  TileLane<HD> lane_at;
  lane_at.init(base);
  const int first = k0 / AT_WALK, tiles = (S + AT_WALK - 1) / AT_WALK;
  auto issue = [&](int t, int buf) {
    issue_tile<HD>(rq, pq, t * AT_WALK, S - 1, base + buf * 2 * TB);
    issue_tile<HD>(rg, pg, t * AT_WALK, S - 1, base + buf * 2 * TB + TB);
    const int q = t * AT_WALK + lane < S ? t * AT_WALK + lane : S - 1;
    if (wave == 0) dma_b32(rl, (uint32_t)q * 4u, sbase + buf * (2 * AT_WALK * 4));
    if (wave == 1) dma_b32(rd, (uint32_t)q * 4u, sbase + buf * (2 * AT_WALK * 4) + AT_WALK * 4);
  };
  issue(first, 0);
  bf16x8_t kf[KS], vf[KS];
  load_own<HD>(rows_of(K), (uint32_t)K.pitch * 2u, w0, S - 1, kf);
  load_own<HD>(rows_of(V), (uint32_t)V.pitch * 2u, w0, S - 1, vf);
  const int my_k = w0 + (lane & 31);
  const float c = scale * LOG2E;
  floatx16_t dk[NB], dv[NB];
#pragma unroll
  for (int d = 0; d < NB; ++d) { dk[d] = zero16(); dv[d] = zero16(); }
  for (int t = first; t < tiles; ++t) {
    const int buf = (t - first) & 1;
    tile_barrier();
    if (t + 1 < tiles) issue(t + 1, buf ^ 1);
    const float* st = stats + buf * 2 * AT_WALK;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int qs = t * AT_WALK + 32 * sub;
      if (qs + 31 < w0) continue;                                       // (the same for the whole wave) every query of it before the wave's keys
      const TileLane<HD> T = lane_at.in(buf * 2 * TB);                  // Q; dO is TB bytes behind
      auto stat_rows = [&](int which) __attribute__((always_inline)) {  // the accumulators start at -lse / scale and -delta
        floatx16_t a;
#pragma unroll
        for (int bq = 0; bq < 4; ++bq) {
          const floatx4_t v = *reinterpret_cast<const floatx4_t*>(st + which * AT_WALK + 32 * sub + 8 * bq + 4 * hi);
#pragma unroll
          for (int j = 0; j < 4; ++j) a[4 * bq + j] = v[j];
        }
        return a;
      };
      floatx16_t s = stat_rows(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = HYC_MFMA(frag_rows<HD>(T, 0, 32 * sub, ks), kf[ks], s);
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(s[i] * c);
      if (qs < w0 + 31 || qs + 31 >= S) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int q = qs + 8 * (i >> 2) + 4 * hi + (i & 3);
          if (q < my_k || q >= S) s[i] = 0.f;
        }
      }
      __builtin_amdgcn_sched_barrier(0);                                // (a phase's fragment reads stay in it: registers)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const bf16x8_t pf = acc_frag(s, half);
#pragma unroll
        for (int d = 0; d < NB; ++d) dv[d] = HYC_MFMA(frag_cols<HD>(T, TB, 32 * d, 32 * sub + 16 * half), pf, dv[d]);
      }
      __builtin_amdgcn_sched_barrier(0);
      floatx16_t dp = stat_rows(1);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        dp = HYC_MFMA(frag_rows<HD>(T, TB, 32 * sub, ks), vf[ks], dp);
        if (ks % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) dp[i] *= s[i];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const bf16x8_t df = acc_frag(dp, half);
#pragma unroll
        for (int d = 0; d < NB; ++d) dk[d] = HYC_MFMA(frag_cols<HD>(T, 0, 32 * d, 32 * sub + 16 * half), df, dk[d]);
      }
    }
  }
#pragma unroll
  for (int d = 0; d < NB; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[d][i] *= scale;
  __syncthreads();
  uint16_t* T = lds + wave * 32 * HD;
  store_own<HD>(dv, T, DV.p + (int64_t)b * S * DV.pitch + (int64_t)h * HD, DV.pitch, w0, S, nullptr, nullptr);
  store_own<HD>(dk, T, DK.p + (int64_t)b * S * DK.pitch + (int64_t)h * HD, DK.pitch, w0, S, cosv, sinv);
}

// What the backward's accumulators start from: -delta, delta[b, h, s] = sum over the head's channels of dO * O (HD / 8
// lanes per token and head), and -lse / scale.
template <int HD>
__global__ void __launch_bounds__(256)
k_attn_delta(AttnRows G, AttnRows O, const float* __restrict__ lse, float* __restrict__ nlse, float* __restrict__ ndelta, int S, int heads,
             int64_t items, float inv_scale) {
  constexpr int L = HD / 8;
  const int64_t it = ((int64_t)blockIdx.x * 256 + threadIdx.x) / L;
  const int c = threadIdx.x % L;
  float v = 0.f;
  const int64_t bs = it / heads;
  const int h = (int)(it - bs * heads);
  if (it < items) {
    float g[8], o[8];
    unpack8(*reinterpret_cast<const uint4*>(G.p + bs * G.pitch + (int64_t)h * HD + 8 * c), g);
    unpack8(*reinterpret_cast<const uint4*>(O.p + bs * O.pitch + (int64_t)h * HD + 8 * c), o);
#pragma unroll
    for (int j = 0; j < 8; ++j) v = __builtin_fmaf(g[j], o[j], v);
  }
  v = group_reduce<L>(v, OpAdd());
  if (c == 0 && it < items) {
    const int64_t b = bs / S, s = bs - b * S;
    const int64_t at = (b * heads + h) * S + s;
    ndelta[at] = -v;
    nlse[at] = -(lse[at] * inv_scale);
  }
}

static int attn_args(const char* who, int64_t B, int64_t S, int64_t heads, int64_t hd, float scale, const int64_t* pitches, int n) {
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

using namespace hyc;

extern "C" {

int hyc_attn_fwd(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv, int64_t B, int64_t S,
                 int64_t heads, int64_t head_dim, float scale, void* out, int64_t ldo, float* lse, void* stream) {
  const int64_t pitches[4] = {ldq, ldk, ldv, ldo};
  int rc = attn_args("hyc_attn_fwd", B, S, heads, head_dim, scale, pitches, 4);
  if (rc) return rc;
  if (B == 0 || S == 0) return HYC_OK;
  if (!q || !k || !v || !out || !lse) return fail(HYC_EFAULT, "hyc_attn_fwd: null buffer");
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out)) return fail(HYC_EINVAL, "hyc_attn_fwd: buffers must be 16-byte aligned");
  hipStream_t st = begin_launch(stream);
  const int blocks = (int)((S + AT_OWN - 1) / AT_OWN), BH = (int)(B * heads);
  const AttnRows Q{(const uint16_t*)q, ldq}, K{(const uint16_t*)k, ldk}, V{(const uint16_t*)v, ldv};
  const AttnOut O{(uint16_t*)out, ldo};
#define HYC_GO(HD_) hipLaunchKernelGGL((k_attn_fwd<HD_>), dim3((unsigned)(blocks * BH)), dim3(256), 0, st, Q, K, V, O, lse, (int)S, (int)heads, BH, blocks, scale)
  if (head_dim == 128) HYC_GO(128);
  else HYC_GO(64);
#undef HYC_GO
  return check_launch("hyc_attn_fwd");
}

int hyc_attn_bwd(const void* dout, int64_t ldg, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv,
                 const void* out, int64_t ldo, const float* lse, const void* cosv, const void* sinv, int64_t B, int64_t S,
                 int64_t heads, int64_t head_dim, float scale, void* dq, int64_t lddq, void* dk, int64_t lddk, void* dv,
                 int64_t lddv, float* workspace, void* stream) {
  const int64_t pitches[8] = {ldg, ldq, ldk, ldv, lddq, lddk, lddv, ldo};
  int rc = attn_args("hyc_attn_bwd", B, S, heads, head_dim, scale, pitches, 8);
  if (rc) return rc;
  if (B == 0 || S == 0) return HYC_OK;
  if (!dout || !q || !k || !v || !out || !lse || !workspace || !dq || !dk || !dv || ((cosv == nullptr) != (sinv == nullptr)))
    return fail(HYC_EFAULT, "hyc_attn_bwd: null buffer");
  if (!aligned16(dout) || !aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out) || !aligned16(dq) || !aligned16(dk) || !aligned16(dv) ||
      (cosv && (!aligned16(cosv) || !aligned16(sinv))))
    return fail(HYC_EINVAL, "hyc_attn_bwd: buffers must be 16-byte aligned");
  hipStream_t st = begin_launch(stream);
  const int blocks = (int)((S + AT_OWN - 1) / AT_OWN), BH = (int)(B * heads);
  const AttnRows Q{(const uint16_t*)q, ldq}, K{(const uint16_t*)k, ldk}, V{(const uint16_t*)v, ldv}, G{(const uint16_t*)dout, ldg};
  const AttnRows O{(const uint16_t*)out, ldo};
  const AttnOut DQ{(uint16_t*)dq, lddq}, DK{(uint16_t*)dk, lddk}, DV{(uint16_t*)dv, lddv};
  const dim3 grid((unsigned)(blocks * BH));
  const int64_t items = B * S * heads;
  float *nlse = workspace, *ndelta = workspace + items;
  const unsigned dgrid = (unsigned)((items * (head_dim / 8) + 255) / 256);
#define HYC_GO(HD_)                                                                                                              \
  do {                                                                                                                           \
    hipLaunchKernelGGL((k_attn_delta<HD_>), dim3(dgrid), dim3(256), 0, st, G, O, lse, nlse, ndelta, (int)S, (int)heads, items,    \
                       1.0f / scale);                                                                                            \
    hipLaunchKernelGGL((k_attn_bwd_dkdv<HD_>), grid, dim3(256), 0, st, Q, K, V, G, nlse, ndelta, (const uint16_t*)cosv,             \
                       (const uint16_t*)sinv, DK, DV, (int)S, (int)heads, BH, blocks, scale);                                    \
    hipLaunchKernelGGL((k_attn_bwd_dq<HD_>), grid, dim3(256), 0, st, Q, K, V, G, nlse, ndelta, (const uint16_t*)cosv,              \
                       (const uint16_t*)sinv, DQ, (int)S, (int)heads, BH, blocks, scale);                                        \
  } while (0)
  if (head_dim == 128) HYC_GO(128);
  else HYC_GO(64);
#undef HYC_GO
  return check_launch("hyc_attn_bwd");
}

}  // extern "C"
