// The rank-r terms of LoRA projections beside a frozen NF4 base (the reference: peft `Linear.forward` around
// bitsandbytes_fix/_function.py:509-540, once per projection), a group of projections of one input at a time:
//
//   forward     h = x A^T;  y = s h B^T, onto which the base product accumulates (the rank-r term is rounded to bf16 before
//               it is added, as it is when it is a tensor of its own)
//   backward    dX = [dY | dh] [W^T | A^T]^T: ONE product over all projections of the group, the rank-r columns as R further
//               columns of its reduction;  dh = s dY B and dB = s dY^T h both from ONE read of dY
//
// The transient weight of the backward is written transposed: the library's GEMMs with both operands contiguous along the
// reduction are 10-20 % faster (dX of a 3 x 4096 group at 4096 tokens: three accumulating products 318 us, one 293, one with
// the transposed weight 252; 2 x 11008: 551 / 525 / 460).
#include <type_traits>

#include "abi_util.hpp"
#include "nf4_levels.hpp"
#include "row_kernels.hpp"

namespace hyc {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
#define HYC_MFMA16(a_, b_, c_) __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_, b_, c_, 0, 0, 0)

constexpr int64_t LORA_WT_WIDE = 512;                   // workgroups from which k_lora_weight_t walks four steps
constexpr int LORA_MAX = 4;                              // projections of a group

struct LoraGroup {
  const uint16_t* f[LORA_MAX];                           // the LoRA factors (A [r, K] or B [out, r])
  int end[LORA_MAX];                                     // first row of the stacked weight after projection i
  int n, r;
};

// out[k, n] = the dequantised W[n, k] for n < rows, A_i[j, k] for n = rows + i r + j, zeros in the rest of the room.  A
// workgroup turns 128 n x 64 STEPS k in LDS, 64 k at a time: a lane decodes weights of two neighbouring n and writes them as
// pairs (64 lanes = consecutive banks), rows of k leave as whole 256-byte runs.
// STEPS = 4: every wave holds one 64-k scale group of its two n (32 bytes of codes each), so that the four waves together
// use whole 128-byte lines of the codes, all requested at the start; with STEPS = 1 a line goes to four workgroups, which
// the dispatcher spreads over four L2s.  The four groups of a 4096-wide layer (202 M weights): 45 -> 31 us each on
// average, 4 TB/s; the groups of a 2048-wide layer, that stay at STEPS = 1 but for one, 12.2 -> 10.9 (codes requested before the table is)
// STEPS = 1 remains where four times fewer workgroups would leave the chip idle.
template <int STEPS>
__global__ void __launch_bounds__(256)
k_lora_weight_t(const uint8_t* __restrict__ packed, const float* __restrict__ absmax, int rows, int K, int room, LoraGroup g,
                uint16_t* __restrict__ out) {
  __shared__ float lut[16];
  __shared__ __align__(16) uint32_t T[64][64 + 4];       // [k][n / 2]
  if (threadIdx.x < 16) lut[threadIdx.x] = kNF4[threadIdx.x];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = blockIdx.y * 128, k0 = blockIdx.x * 64 * STEPS, N = rows + room;
  const int64_t pitch = N;
  const int kw = k0 + 16 * STEPS * wave;                 // this wave's k: 16 of them per step
  const bool on = kw < K;                                // (K is a multiple of 64)
  uint2 code[2][STEPS];
  float scale[2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int n = n0 + 2 * lane + a;
    scale[a] = 0.f;
#pragma unroll
    for (int t = 0; t < STEPS; ++t) code[a][t] = make_uint2(0, 0);
    if (on && n < rows) {
      const int64_t at = (int64_t)n * K + kw;
      scale[a] = absmax[at >> 6];
      if (STEPS == 4) {
        const uint4 lo = *reinterpret_cast<const uint4*>(packed + at / 2), hi = *reinterpret_cast<const uint4*>(packed + at / 2 + 16);
        code[a][0] = make_uint2(lo.x, lo.y); code[a][1 % STEPS] = make_uint2(lo.z, lo.w);
        code[a][2 % STEPS] = make_uint2(hi.x, hi.y); code[a][3 % STEPS] = make_uint2(hi.z, hi.w);
      } else {
        code[a][0] = *reinterpret_cast<const uint2*>(packed + at / 2);
      }
    }
  }
  __syncthreads();                                       // the table
#pragma unroll
  for (int t = 0; t < STEPS; ++t) {
    float v[2][16];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const int n = n0 + 2 * lane + a;
      if (n < rows) {
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const uint32_t byte = ((b < 4 ? code[a][t].x : code[a][t].y) >> (8 * (b & 3))) & 0xFFu;
          v[a][2 * b] = lut[byte >> 4] * scale[a];
          v[a][2 * b + 1] = lut[byte & 15u] * scale[a];
        }
      } else {
        const int f = n - rows, p = f / g.r;
#pragma unroll
        for (int j = 0; j < 16; ++j) v[a][j] = 0.f;
        if (on && p < g.n) {
          const uint16_t* A = g.f[p] + (int64_t)(f - p * g.r) * K + kw + 16 * t;
          float lo[8], hi[8];
          unpack8(*reinterpret_cast<const uint4*>(A), lo);
          unpack8(*reinterpret_cast<const uint4*>(A + 8), hi);
#pragma unroll
          for (int j = 0; j < 8; ++j) { v[a][j] = lo[j]; v[a][8 + j] = hi[j]; }
        }
      }
    }
    if (t) __syncthreads();                              // the previous step has left the tile
#pragma unroll
    for (int j = 0; j < 16; ++j) T[16 * wave + j][lane] = pack_bf16(v[0][j], v[1][j]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int at = threadIdx.x + 256 * u, r = at / 16, c = at % 16;
      const int k = k0 + 16 * STEPS * (r / 16) + 16 * t + r % 16;       // tile row r = wave r / 16, its k number r % 16
      if (k < K && n0 + 8 * c < N)
        *reinterpret_cast<uint4*>(out + (int64_t)k * pitch + n0 + 8 * c) = *reinterpret_cast<const uint4*>(&T[r][4 * c]);
    }
  }
}

// h[m, i r + j] = sum_k x[m, k] A_i[j, k].  Eight waves share 16 tokens, each taking every eighth block of 64 channels; A stays
// in L2.  Should be bound by the read of x (4096 x 4096: 33.5 MB).  Loading the operands of the products straight from memory
// puts neighbouring lanes into different rows, which the load path takes far longer for than for whole lines: 4 us per 16 columns
// of h, however many tokens there are (and however many loads are under way).  So a wave loads 16 rows x 128 bytes as lines and turns them in 2 KB of LDS of
// its own (no barrier: a wave's LDS operations are in order); the swizzle puts the 16 lanes of a read and of a write on all
// banks.  4096 x 4096 with 16 / 32 / 48 columns 10.9 / 15.5 / 19.6 -> 8.4 / 12.2 / 14.8 us, 4096 x 11008 with 16 31.4 -> 26.0 (2048 tokens: 10.9 / 15.2 /
// 19.4 / 27.6 -> 8.2 / 10.8 / 13.5 / 18.5).  Starting every workgroup at another block gave 5 % more at most, for sums that depend
// on a token's place in the batch: not taken.
template <int CT>
__global__ void __launch_bounds__(512, 2)
k_lora_down(const uint16_t* __restrict__ x, int64_t ldx, int64_t M, int K, LoraGroup g, uint16_t* __restrict__ h) {
  constexpr int TILE = 16 * 64;                          // 16 rows of 64 channels
  __shared__ __align__(16) uint16_t lds[8][(1 + CT) * TILE];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l15 = lane & 15, lq = lane >> 4;
  const int64_t m0 = (int64_t)blockIdx.x * 16;
  const int nr = g.n * g.r, lr = lane >> 3, lc = lane & 7;   // a load brings eight rows of eight chunks
  const uint16_t *xp[2], *ap[CT][2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int64_t m = m0 + 8 * u + lr < M ? m0 + 8 * u + lr : M - 1;
    xp[u] = x + m * ldx + 8 * lc;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int f = 16 * c + 8 * u + lr, ff = f < nr ? f : 0, p = ff / g.r;
      ap[c][u] = g.f[p] + (int64_t)(ff - p * g.r) * K + 8 * lc;
    }
  }
  floatx4_t acc[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) acc[c] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int U = CT == 1 ? 8 : CT <= 3 ? 4 : 2;       // blocks whose loads are under way together (at most 128 registers)
  const int blocks = K / 64;
  uint16_t* T = lds[wave];
  auto run = [&](int s, auto uno) __attribute__((always_inline)) {
    constexpr int UU = decltype(uno)::value;
    bf16x8_t a[UU][2], b[UU][CT][2];
#pragma unroll
    for (int u = 0; u < UU; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[u][i] = *reinterpret_cast<const bf16x8_t*>(xp[i] + 64 * (s + 8 * u));
#pragma unroll
        for (int c = 0; c < CT; ++c) b[u][c][i] = *reinterpret_cast<const bf16x8_t*>(ap[c][i] + 64 * (s + 8 * u));
      }
    __builtin_amdgcn_sched_barrier(0);                   // (the scheduler would trade loads in flight for occupancy)
#pragma unroll
    for (int u = 0; u < UU; ++u) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = 8 * i + lr, at = row * 64 + 8 * (lc ^ ((row >> 1) & 7));
        *reinterpret_cast<bf16x8_t*>(T + at) = a[u][i];
#pragma unroll
        for (int c = 0; c < CT; ++c) *reinterpret_cast<bf16x8_t*>(T + (1 + c) * TILE + at) = b[u][c][i];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int at = l15 * 64 + 8 * ((4 * ks + lq) ^ ((l15 >> 1) & 7));
        const bf16x8_t av = *reinterpret_cast<const bf16x8_t*>(T + at);
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[c] = HYC_MFMA16(av, *reinterpret_cast<const bf16x8_t*>(T + (1 + c) * TILE + at), acc[c]);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  };
  int s = wave;
  for (; s + 8 * (U - 1) < blocks; s += 8 * U) run(s, std::integral_constant<int, U>{});
  if constexpr (U > 4)
    if (s + 8 * 3 < blocks) { run(s, std::integral_constant<int, 4>{}); s += 8 * 4; }
  if constexpr (U > 2)
    if (s + 8 < blocks) { run(s, std::integral_constant<int, 2>{}); s += 8 * 2; }
  if (s < blocks) run(s, std::integral_constant<int, 1>{});
  // the waves' sums meet in the same memory: a wave's CT * 256 floats fit its own tiles
  float* red = reinterpret_cast<float*>(T);
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[c * 256 + (4 * lq + i) * 16 + l15] = acc[c][i];
  __syncthreads();
  for (int e = threadIdx.x; e < 16 * nr; e += 512) {
    const int t = e / nr, f = e - t * nr;
    if (m0 + t >= M) break;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) sum += reinterpret_cast<const float*>(lds[w])[(f >> 4) * 256 + t * 16 + (f & 15)];
    h[(m0 + t) * nr + f] = f_to_bf(sum);
  }
}

// ---- y = s h B^T ----------------------------------------------------------------------------------------------------
struct LoraOut {
  const uint16_t* B[LORA_MAX];                           // [n_out_i, r]
  int n_out[LORA_MAX], fb0[LORA_MAX + 1], row0[LORA_MAX + 1];   // first feature block / first column of projection i
  int n, r;
};
constexpr int LO_F = 256, LO_M = 128;                    // features and tokens of a workgroup

// A pure write (4096 tokens x 12288: 100 MB), so the point is full 16-byte stores: the products are taken with the features
// as rows in the order that gives a lane eight neighbouring features of its token over two MFMAs.  Ordinary stores: the base
// product reads y next, from the last-level cache.
__global__ void __launch_bounds__(256)
k_lora_up(const uint16_t* __restrict__ h, int64_t M, LoraOut a, float scale, uint16_t* __restrict__ y) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l15 = lane & 15, lq = lane >> 4;
  int p = 0;
  while (p + 1 < a.n && (int)blockIdx.x >= a.fb0[p + 1]) ++p;
  const int f0 = ((int)blockIdx.x - a.fb0[p]) * LO_F + 64 * wave, r = a.r, nr = a.n * r, n_out = a.n_out[p];
  const int64_t m_begin = (int64_t)blockIdx.y * LO_M, pitch = a.row0[a.n];
  const bool on = 8 * lq < r;                            // (r is a multiple of 8)
  bf16x8_t bf[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int f = f0 + 32 * (q >> 1) + 8 * (l15 >> 2) + 4 * (q & 1) + (l15 & 3);
    const uint4 v = on && f < n_out ? *reinterpret_cast<const uint4*>(a.B[p] + (int64_t)f * r + 8 * lq) : make_uint4(0, 0, 0, 0);
    bf[q] = __builtin_bit_cast(bf16x8_t, v);
  }
#pragma unroll 4
  for (int t = 0; t < LO_M; t += 16) {
    const int64_t m = m_begin + t + l15;
    const uint4 v = on && m < M ? *reinterpret_cast<const uint4*>(h + m * nr + p * r + 8 * lq) : make_uint4(0, 0, 0, 0);
    const bf16x8_t hf = __builtin_bit_cast(bf16x8_t, v);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const floatx4_t z = {0.f, 0.f, 0.f, 0.f};
      const floatx4_t d0 = HYC_MFMA16(bf[2 * g], hf, z), d1 = HYC_MFMA16(bf[2 * g + 1], hf, z);
      const int f = f0 + 32 * g + 8 * lq;
      if (m < M && f < n_out) {
        const float o[8] = {d0[0] * scale, d0[1] * scale, d0[2] * scale, d0[3] * scale, d1[0] * scale, d1[1] * scale, d1[2] * scale, d1[3] * scale};
        *reinterpret_cast<uint4*>(y + m * pitch + a.row0[p] + f) = pack8(o);
      }
    }
  }
}

// ---- dx = g w for a weight of few rows -------------------------------------------------------------------------------------
// dx[m, k] = sum_j g[m, j] w[j, k], j < N <= 32.  A pure write like k_lora_up, and laid out like it; what differs is the weight, whose
// columns are the features here: a lane gathers the 8 rows of its feature (2 bytes each, 64-byte runs over the lanes, once per
// 128 tokens, from L2).
__global__ void __launch_bounds__(256)
k_thin_dx(const uint16_t* __restrict__ g, int64_t ldg, int64_t M, const uint16_t* __restrict__ w, int N, int K, uint16_t* __restrict__ dx) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l15 = lane & 15, lq = lane >> 4;
  const int f0 = (int)blockIdx.x * LO_F + 64 * wave;
  const int64_t m_begin = (int64_t)blockIdx.y * LO_M;
  const bool on = 8 * lq < N;                            // (N is a multiple of 8)
  bf16x8_t wf[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int f = f0 + 32 * (q >> 1) + 8 * (l15 >> 2) + 4 * (q & 1) + (l15 & 3);
#pragma unroll
    for (int j = 0; j < 8; ++j) wf[q][j] = __builtin_bit_cast(__bf16, on && f < K ? w[(int64_t)(8 * lq + j) * K + f] : (uint16_t)0);
  }
#pragma unroll 4
  for (int t = 0; t < LO_M; t += 16) {
    const int64_t m = m_begin + t + l15;
    const uint4 v = on && m < M ? *reinterpret_cast<const uint4*>(g + m * ldg + 8 * lq) : make_uint4(0, 0, 0, 0);
    const bf16x8_t gf = __builtin_bit_cast(bf16x8_t, v);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const floatx4_t z = {0.f, 0.f, 0.f, 0.f};
      const floatx4_t d0 = HYC_MFMA16(wf[2 * c], gf, z), d1 = HYC_MFMA16(wf[2 * c + 1], gf, z);
      const int f = f0 + 32 * c + 8 * lq;
      if (m < M && f < K) {
        const float o[8] = {d0[0], d0[1], d0[2], d0[3], d1[0], d1[1], d1[2], d1[3]};
        *reinterpret_cast<uint4*>(dx + m * K + f) = pack8(o);
      }
    }
  }
}

// ---- dh = s dY B and dB = s dY^T h from one read of dY -----------------------------------------------------------------
struct LoraUp {
  const uint16_t* g[LORA_MAX];                           // dY_i [M, n_out_i], rows ldg_i apart
  int64_t ldg[LORA_MAX];
  const uint16_t* B[LORA_MAX];                           // [n_out_i, r]
  uint16_t* dB[LORA_MAX];
  int n_out[LORA_MAX], fb0[LORA_MAX + 1], row0[LORA_MAX + 1];   // first feature block / first stacked row of projection i
  int n, r;
};
constexpr int LU_F = 256, LU_M = 32;                     // features of a workgroup, tokens of a tile

__device__ __forceinline__ int lu_swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }

// A workgroup owns 256 features and a range of tokens, walked in tiles of 32 that go from memory straight to LDS, NB of them
// under way (two workgroups per CU).  From a tile, wave w takes the 64 features 64 w .. for both products: dY rows as stored
// are the operand of dh (the wave's part of B in registers), the transposing read gives that of dB.  The waves' sums for dh meet in
// LDS.  dh leaves as one fp32 partial per feature block, dB as one per token range; k_lora_up_finish adds them in a fixed order.
//
// The read of dY bounds it, so nothing may empty the queue of loads: every memory operation of the walk is unconditional (what
// lies outside its resource is dropped, or reads zeros) and a wave waits for its oldest tile by count, over the stores behind it.
// Both launches at 4096 tokens x 4096 with the copy / 3 x 4096 / 2 x 11008 features: 25.9 / 33.8 / 49.4 -> 21.8 / 26.6 / 40.5 us against two
// buffers of 64 tokens, waited for with the stores, and a grid that was a little more than resident (2048 tokens: 16.9 / 25.8 / 31.3 -> 14.3 /
// 18.7 / 27.9; 157 tokens x 2048 / 3 x 2048 / 2 x 5632: 10.8 / 10.9 / 11.7 -> 8.3 / 9.2 / 8.8).  dY then arrives at up to 4.9 TB/s.
template <int RT, bool COPY>
__global__ void __launch_bounds__(256, 2)
k_lora_up_bwd(LoraUp a, int64_t M, const uint16_t* __restrict__ h, int tokens, float* __restrict__ dhp, float* __restrict__ dbp,
              uint16_t* __restrict__ copy, int64_t ld_copy) {
  constexpr int RC = 16 * RT;                            // columns of the factor, padded
  constexpr int NB = RT == 1 ? 4 : 3;                    // (76 and 70 KB of LDS)
  constexpr int S = COPY ? 5 : 1;                        // stores of a wave per tile
  __shared__ __align__(1024) uint16_t tile[NB][LU_M * LU_F];
  __shared__ __align__(1024) uint16_t ht[NB][LU_M * RC];
  __shared__ __align__(16) float red[4][LU_M * RC];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l15 = lane & 15, lq = lane >> 4;
  const int fb = blockIdx.x;
  int p = 0;
  while (p + 1 < a.n && fb >= a.fb0[p + 1]) ++p;
  const int f0 = (fb - a.fb0[p]) * LU_F, n_out = a.n_out[p], r = a.r, nr = a.n * r;
  const int64_t m_begin = (int64_t)blockIdx.y * tokens, m_end = m_begin + tokens < M ? m_begin + tokens : M;
  const int count = (int)(m_end - m_begin), tiles = (count + LU_M - 1) / LU_M;
  const uint32_t pitch = (uint32_t)a.ldg[p] * 2u;
  const uint16_t* base = a.g[p] + m_begin * a.ldg[p] + f0;
  // (the resources end with the last row's last feature of this block: tokens past the range and features past the end are zeros)
  const int fl = n_out - f0 < LU_F ? n_out - f0 : LU_F;  // features this block really has, a multiple of 8
  const u32x4_t rs = uniform_rsrc(base, (uint32_t)(count - 1) * pitch + 2u * (uint32_t)fl);
  const u32x4_t rs_h = uniform_rsrc(h + m_begin * nr + p * r, 2u * ((uint32_t)(count - 1) * (uint32_t)nr + (uint32_t)r));
  const uint32_t lds_t = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)&tile[0][0];
  const uint32_t lds_h = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)&ht[0][0];
  const int ir = lane >> 5, ic = lane & 31;              // an instruction brings two rows of 32 chunks
  // (the chunk at position ic of row 2 (wave + 4 u) + ir is ic ^ swz(row); swz has a period of 16 rows: that of u + 2)
  uint32_t vt[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int row = 2 * (wave + 4 * u) + ir, c = ic ^ lu_swz(row & 15);
    vt[u] = 8 * c < fl ? (uint32_t)row * pitch + 16u * (uint32_t)c : NOWHERE;
  }
  const int hrow = (wave * 64 + lane) / (RC / 8), hcol = 8 * ((wave * 64 + lane) % (RC / 8));   // (the first RT waves bring the rows of h)
  const uint32_t vh = hcol < r ? 2u * ((uint32_t)hrow * (uint32_t)nr + (uint32_t)hcol) : NOWHERE;
  auto issue = [&](int t, int buf) __attribute__((always_inline)) {
    const uint32_t at = (uint32_t)(t * LU_M) * pitch;
#pragma unroll
    for (int u = 0; u < 4; ++u) dma_b128(rs, vt[u] == NOWHERE ? NOWHERE : vt[u] + at, lds_t + (uint32_t)(buf * LU_M * LU_F * 2 + (wave + 4 * u) * 1024));
    if (wave < RT)
      dma_b128(rs_h, vh == NOWHERE ? NOWHERE : vh + (uint32_t)(t * LU_M) * 2u * (uint32_t)nr, lds_h + (uint32_t)(buf * LU_M * RC * 2 + wave * 1024));
  };
  // tile t has landed.  Behind its loads in the queue are those of up to NB - 1 further tiles and the stores of as many steps (at the
  // start and the end of the walk the loads alone are counted: the stores then only make the wait longer than it need be)
  auto landed = [&](int t) __attribute__((always_inline)) {
    const int ahead = tiles - 1 - t < NB - 1 ? tiles - 1 - t : NB - 1;
#define HYC_WAIT(L_)                                                                                                         \
    do {                                                                                                                     \
      if (ahead == NB - 1 && t >= NB - 1) asm volatile("s_waitcnt vmcnt(%0)" :: "n"((NB - 1) * (L_ + S)) : "memory");         \
      else if (ahead == 3) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(3 * L_) : "memory");                                    \
      else if (ahead == 2) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * L_) : "memory");                                    \
      else if (ahead == 1) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(L_) : "memory");                                        \
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                                                  \
    } while (0)
    if (wave < RT) HYC_WAIT(5);
    else HYC_WAIT(4);
#undef HYC_WAIT
  };
  // (LDS operations only: __syncthreads may wait for the loads and stores under way)
  auto meet = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
#pragma unroll
  for (int t = 0; t < NB; ++t)
    if (t < tiles) issue(t, t);
  // B as the first operand of dh^T: lane = column l % 16, 8 consecutive features per reduction step
  bf16x8_t bf[2][RT];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int f = f0 + 64 * wave + 32 * ks + 8 * lq + j, c = 16 * rt + l15;
        const uint16_t v = f < n_out && c < r ? a.B[p][(int64_t)f * r + c] : (uint16_t)0;
        bf[ks][rt][j] = __builtin_bit_cast(__bf16, v);
      }
  floatx4_t db[4][RT];
#pragma unroll
  for (int ft = 0; ft < 4; ++ft)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) db[ft][rt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  typedef bf16x4_t __attribute__((address_space(3))) * lds_b64;
  auto tr8 = [](const uint16_t* q0, const uint16_t* q1) __attribute__((always_inline)) {
    const bf16x4_t x = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_b64)const_cast<uint16_t*>(q0));
    const bf16x4_t y = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_b64)const_cast<uint16_t*>(q1));
    bf16x8_t f;
    f[0] = x[0]; f[1] = x[1]; f[2] = x[2]; f[3] = x[3]; f[4] = y[0]; f[5] = y[1]; f[6] = y[2]; f[7] = y[3];
    return f;
  };
  const BufferRsrc rs_dh = make_rsrc(dhp + ((int64_t)fb * M + m_begin) * RC, (uint32_t)count * RC * 4u);
  int buf = 0;
  for (int t = 0; t < tiles; ++t) {
    landed(t);
    meet();
    const uint16_t* T = tile[buf];
    if constexpr (COPY) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int row0 = 2 * wave + 8 * u, left = count - t * LU_M - row0, c = ic ^ lu_swz((row0 + ir) & 15);
        const BufferRsrc rs_c = make_rsrc(copy + (m_begin + t * LU_M + row0) * ld_copy + a.row0[p] + f0,
                                          left > 0 ? 2u * ((left > 1 ? (uint32_t)ld_copy : 0u) + (uint32_t)fl) : 0u);
        const uint4 v = *reinterpret_cast<const uint4*>(T + (row0 + ir) * LU_F + 8 * ic);
        const u32x4_t w = {v.x, v.y, v.z, v.w};
        __builtin_amdgcn_raw_buffer_store_b128(w, rs_c, (int)(8 * c < fl ? (ir ? 2u * (uint32_t)ld_copy : 0u) + 16u * (uint32_t)c : NOWHERE), 0, 0);
      }
    }
#pragma unroll
    for (int tg = 0; tg < 2; ++tg) {
      floatx4_t dh[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) dh[rt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16x8_t x = *reinterpret_cast<const bf16x8_t*>(T + (16 * tg + l15) * LU_F + 8 * ((8 * wave + 4 * ks + lq) ^ lu_swz(l15)));
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) dh[rt] = HYC_MFMA16(bf[ks][rt], x, dh[rt]);
      }
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) *reinterpret_cast<floatx4_t*>(&red[wave][(16 * tg + l15) * RC + 16 * rt + 4 * lq]) = dh[rt];
    }
    {
      const int r0 = 8 * lq + (l15 >> 2), r1 = r0 + 4;
      bf16x8_t hb[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const uint16_t* q = &ht[buf][16 * rt + 4 * (l15 & 3)];
        hb[rt] = tr8(q + r0 * RC, q + r1 * RC);
      }
#pragma unroll
      for (int ft = 0; ft < 4; ++ft) {
        const int col = 64 * wave + 16 * ft + 4 * (l15 & 3);
        const bf16x8_t x = tr8(T + r0 * LU_F + 8 * ((col >> 3) ^ lu_swz(r0 & 15)) + (col & 7),
                               T + r1 * LU_F + 8 * ((col >> 3) ^ lu_swz(r1 & 15)) + (col & 7));
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) db[ft][rt] = HYC_MFMA16(x, hb[rt], db[ft][rt]);
      }
    }
    meet();
    if (t + NB < tiles) issue(t + NB, buf);
    {
      typedef float sum_t __attribute__((ext_vector_type(2 * RT)));
      const int e = 2 * RT * threadIdx.x;
      sum_t s = *reinterpret_cast<const sum_t*>(&red[0][e]);
#pragma unroll
      for (int w = 1; w < 4; ++w) s += *reinterpret_cast<const sum_t*>(&red[w][e]);
      const uint32_t off = 4u * (uint32_t)(t * LU_M * RC + e);
      if constexpr (RT == 1) {
        const u32x2_t w = __builtin_bit_cast(u32x2_t, s);    // (the whole vector: a bit cast of one element reads the first)
        store_b64(rs_dh, off, w.x, w.y);
      } else {
        const u32x4_t w = __builtin_bit_cast(u32x4_t, s);
        __builtin_amdgcn_raw_buffer_store_b128(w, rs_dh, (int)off, 0, 0);
      }
    }
    buf = buf + 1 < NB ? buf + 1 : 0;
  }
  float* o = dbp + ((int64_t)blockIdx.y * a.row0[a.n] + a.row0[p] + f0) * RC;
#pragma unroll
  for (int ft = 0; ft < 4; ++ft)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int f = 64 * wave + 16 * ft + 4 * lq + i;
      if (f < fl) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) o[(int64_t)f * RC + 16 * rt + l15] = db[ft][rt][i];
      }
    }
}

// s = in[0] + in[stride] + ... (n terms, in that order), 16 of them requested at a time: the walk over the partial results is
// a chain of latencies
__device__ __forceinline__ float lora_sum(const float* __restrict__ in, int64_t stride, int n) {
  float s = 0.f;
  for (int t = 0; t < n; t += 16) {
    float v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = t + u < n ? in[(t + u) * stride] : 0.f;
#pragma unroll
    for (int u = 0; u < 16; ++u) s += v[u];
  }
  return s;
}

// Adds the partial results: dh (scaled, bf16) to dh [M, n r] and to the columns behind the dY in ext, zeros behind those, dB to
// each dB_i.  A workgroup takes 256 / RC tokens of one projection, or as many rows of the stacked B: the RC columns of a
// partial row lie side by side, so a wave reads whole runs of 256 bytes.
// At 4096 tokens x 4096 / 3 x 4096 / 2 x 11008 features 10.6 / 9.0 / 15.3 -> 4.8 / 6.0 / 7.0 us against a thread per column of the
// room that walked the partial rows one load after the other.
template <int RC>
__global__ void __launch_bounds__(256)
k_lora_up_finish(LoraUp a, int64_t M, const float* __restrict__ dhp, const float* __restrict__ dbp, int ranges, float scale,
                 uint16_t* __restrict__ dh, uint16_t* __restrict__ tail, int64_t ld_tail, int room, unsigned token_blocks) {
  constexpr int ROWS = 256 / RC;
  const int nr = a.n * a.r, j = threadIdx.x & (RC - 1), sub = threadIdx.x / RC;
  if (blockIdx.x < token_blocks * (unsigned)a.n) {
    const int p = (int)(blockIdx.x / token_blocks);
    const int64_t m = (int64_t)(blockIdx.x - p * token_blocks) * ROWS + sub;
    if (m >= M) return;
    uint16_t* row = tail + m * ld_tail;
    if (j < a.r) {
      const int f0 = a.fb0[p];
      const uint16_t v = f_to_bf(lora_sum(dhp + ((int64_t)f0 * M + m) * RC + j, M * RC, a.fb0[p + 1] - f0) * scale);
      dh[m * nr + p * a.r + j] = v;
      row[p * a.r + j] = v;
    }
    if (p == 0)
      for (int c = nr + 8 * j; c < room; c += 8 * RC) *reinterpret_cast<uint4*>(row + c) = make_uint4(0, 0, 0, 0);
    return;
  }
  const int64_t row = (int64_t)(blockIdx.x - token_blocks * (unsigned)a.n) * ROWS + sub;
  const int rows = a.row0[a.n];
  if (row >= rows || j >= a.r) return;
  int p = 0;
  while (p + 1 < a.n && row >= a.row0[p + 1]) ++p;
  a.dB[p][(row - a.row0[p]) * a.r + j] = f_to_bf(lora_sum(dbp + row * RC + j, (int64_t)rows * RC, ranges) * scale);
}

static int lora_group(const char* who, const void* const* factors, const int64_t* n_out, int32_t n, int32_t r, int64_t K, LoraGroup* g) {
  if (n < 1 || n > LORA_MAX) return fail(HYC_ENOTSUP, "%s: %d projections (1 to %d)", who, n, LORA_MAX);
  if (r < 8 || r > 32 || r % 8 != 0) return fail(HYC_ENOTSUP, "%s: rank %d (8, 16, 24 or 32)", who, r);
  if (K <= 0 || K % 64 != 0 || K > (1 << 24)) return fail(HYC_ENOTSUP, "%s: %lld input features (a multiple of 64)", who, (long long)K);
  if (!factors || !n_out) return fail(HYC_EFAULT, "%s: null buffer", who);
  int64_t at = 0;
  for (int i = 0; i < n; ++i) {
    if (!factors[i]) return fail(HYC_EFAULT, "%s: null factor", who);
    if (!aligned16(factors[i])) return fail(HYC_EINVAL, "%s: factors must be 16-byte aligned", who);
    if (n_out[i] <= 0 || n_out[i] % 8 != 0) return fail(HYC_ENOTSUP, "%s: %lld output features (a multiple of 8)", who, (long long)n_out[i]);
    at += n_out[i];
    if (at > (1 << 24)) return fail(HYC_ENOTSUP, "%s: too many output features", who);
    g->f[i] = static_cast<const uint16_t*>(factors[i]);
    g->end[i] = (int)at;
  }
  for (int i = n; i < LORA_MAX; ++i) { g->f[i] = nullptr; g->end[i] = (int)at; }
  g->n = n; g->r = r;
  return HYC_OK;
}

// Token ranges of k_lora_up_bwd, whole tiles each.  512 workgroups are resident at once, two per CU: of the ranges that make a
// workgroup's share of the walk shortest, rounds included, the fewest (each is one more partial dB).  A workgroup's start and end
// count as LU_FIXED tiles.  One workgroup too many is a round of its own: us with 10 / 12 ranges of 4096 x 3 x 4096 26.8 / 31.2, with
// 5 / 6 of 4096 x 2 x 11008 40.6 / 47.4.  At most 32, unless that leaves a range more than 32768 tokens (its offsets into dY are
// 31-bit numbers of bytes up to row pitches of 32760).  Where the rows of dY are so far apart (`pitch` elements) that such a range
// would not fit its 31 bits, as many ranges as it takes workgroups to reach 512, which may be one more.
constexpr int64_t LU_FIXED = 3, LU_RANGE = (int64_t)1 << 30;     // (elements)
static int64_t lora_up_tokens(int64_t M, int64_t fblocks, int64_t pitch) {
  const int64_t tiles = (M + LU_M - 1) / LU_M, least = (M + 32767) / 32768;
  int64_t best = 0, best_cost = 0;
  for (int64_t n = 1; n <= 32 && n <= tiles; ++n) {
    const int64_t each = (tiles + n - 1) / n, used = (tiles + each - 1) / each, cost = (fblocks * used + 511) / 512 * (each + LU_FIXED);
    if (!best || cost < best_cost) { best = each; best_cost = cost; }
  }
  int64_t most = least > 0 ? (tiles + least - 1) / least : 1;
  if (best < most) most = best > 0 ? best : 1;
  if (LU_M * most * pitch >= LU_RANGE) {
    int64_t n = (512 + fblocks - 1) / fblocks;
    if (n > 32) n = 32;
    const int64_t each = (tiles + n - 1) / n;
    if (each > 0 && each < most) most = each;
  }
  return LU_M * most;
}
// partial results of dB a call may have: either rule's
static int64_t lora_up_ranges(int64_t M, int64_t fblocks) {
  const int64_t tokens = lora_up_tokens(M, fblocks, LU_RANGE);
  return M > 0 ? (M + tokens - 1) / tokens : 1;
}
static int lora_up_blocks(const int64_t* n_out, int n) {
  int64_t b = 0;
  for (int i = 0; i < n; ++i) b += (n_out[i] + LU_F - 1) / LU_F;
  return (int)b;
}

}  // namespace hyc

using namespace hyc;

extern "C" {

int hyc_lora_weight_t(const void* packed, const float* absmax, int64_t K, const void* const* A, const int64_t* n_out, int32_t n,
                      int32_t r, int64_t room, void* out, void* stream) {
  LoraGroup g;
  int rc = lora_group("hyc_lora_weight_t", A, n_out, n, r, K, &g);
  if (rc) return rc;
  if (room < (int64_t)n * r || room % 8 != 0 || room > 4096) return fail(HYC_EINVAL, "hyc_lora_weight_t: room=%lld for %d columns", (long long)room, n * r);
  if (!packed || !absmax || !out) return fail(HYC_EFAULT, "hyc_lora_weight_t: null buffer");
  if (!aligned16(packed) || !aligned16(out)) return fail(HYC_EINVAL, "hyc_lora_weight_t: packed and out must be 16-byte aligned");
  const int rows = g.end[n - 1];
  if ((rows + room + 127) / 128 > 65535) return fail(HYC_ENOTSUP, "hyc_lora_weight_t: too many output features");
  hipStream_t st = begin_launch(stream);
  const int64_t down = (rows + room + 127) / 128;
  if ((K + 255) / 256 * down >= LORA_WT_WIDE)
    hipLaunchKernelGGL(k_lora_weight_t<4>, dim3((unsigned)((K + 255) / 256), (unsigned)down), dim3(256), 0, st,
                       static_cast<const uint8_t*>(packed), absmax, rows, (int)K, (int)room, g, static_cast<uint16_t*>(out));
  else
    hipLaunchKernelGGL(k_lora_weight_t<1>, dim3((unsigned)(K / 64), (unsigned)down), dim3(256), 0, st,
                       static_cast<const uint8_t*>(packed), absmax, rows, (int)K, (int)room, g, static_cast<uint16_t*>(out));
  return check_launch("hyc_lora_weight_t");
}

int hyc_lora_down(const void* x, int64_t ldx, int64_t M, int64_t K, const void* const* A, int32_t n, int32_t r, void* h, void* stream) {
  LoraGroup g;
  const int64_t ones[LORA_MAX] = {8, 8, 8, 8};
  int rc = lora_group("hyc_lora_down", A, ones, n, r, K, &g);
  if (rc) return rc;
  const int nr = n * r;
  if (M < 0 || ldx < K || ldx % 8 != 0) return fail(HYC_EINVAL, "hyc_lora_down: M=%lld, row pitch %lld", (long long)M, (long long)ldx);
  if (nr > 96) return fail(HYC_ENOTSUP, "hyc_lora_down: %d columns (at most 96)", nr);
  if (M == 0) return HYC_OK;
  if (!x || !h) return fail(HYC_EFAULT, "hyc_lora_down: null buffer");
  if (!aligned16(x)) return fail(HYC_EINVAL, "hyc_lora_down: x must be 16-byte aligned");
  hipStream_t st = begin_launch(stream);
  const dim3 grid((unsigned)((M + 15) / 16));
#define HYC_GO(CT_)                                                                                                        \
  hipLaunchKernelGGL((k_lora_down<CT_>), grid, dim3(512), 0, st, static_cast<const uint16_t*>(x), ldx, M, (int)K, g,       \
                     static_cast<uint16_t*>(h))
  switch ((nr + 15) / 16) {
    case 1: HYC_GO(1); break;
    case 2: HYC_GO(2); break;
    case 3: HYC_GO(3); break;
    case 4: HYC_GO(4); break;
    case 5: HYC_GO(5); break;
    default: HYC_GO(6); break;
  }
#undef HYC_GO
  return check_launch("hyc_lora_down");
}

int hyc_lora_up(const void* h, int64_t M, const void* const* B, const int64_t* n_out, int32_t n, int32_t r, float scale, void* y,
                void* stream) {
  LoraGroup g;
  int rc = lora_group("hyc_lora_up", B, n_out, n, r, 64, &g);
  if (rc) return rc;
  if (M < 0) return fail(HYC_EINVAL, "hyc_lora_up: M=%lld", (long long)M);
  if (M == 0) return HYC_OK;
  if (!h || !y) return fail(HYC_EFAULT, "hyc_lora_up: null buffer");
  if (!aligned16(h) || !aligned16(y)) return fail(HYC_EINVAL, "hyc_lora_up: buffers must be 16-byte aligned");
  if ((M + LO_M - 1) / LO_M > 65535) return fail(HYC_ENOTSUP, "hyc_lora_up: too many tokens");
  LoraOut a = {};
  a.n = n; a.r = r;
  for (int i = 0; i < n; ++i) {
    a.B[i] = g.f[i];
    a.n_out[i] = (int)n_out[i];
    a.fb0[i + 1] = a.fb0[i] + (int)((n_out[i] + LO_F - 1) / LO_F);
    a.row0[i + 1] = a.row0[i] + (int)n_out[i];
  }
  hipLaunchKernelGGL(k_lora_up, dim3((unsigned)a.fb0[n], (unsigned)((M + LO_M - 1) / LO_M)), dim3(256), 0, begin_launch(stream),
                     static_cast<const uint16_t*>(h), M, a, scale, static_cast<uint16_t*>(y));
  return check_launch("hyc_lora_up");
}

// Where a linear layer of few output features takes k_lora_down and k_thin_dx instead of library products (us, library -> these):
//   x w^T   4096 x 4096 with 8 / 16 / 32 features 11.6 / 12.1 / 9.8 -> 5.7 / 6.0 / 8.6, 4096 x 11008 26.4 / 27.1 / 22.4 -> 17.0 / 17.5 / 20.6,
//           157 x 4096 7.9 / 7.9 / 7.4 -> 4.9 / 5.0 / 7.1; where x no longer stays in the last-level cache the waves' 128-byte rows fall
//           behind: 16384 x 4096 21.8 / 22.0 / 22.6 -> 22.6 / 23.0 / 30.4, 9000 x 13824 37.9 / 39.0 / 41.2 -> 43.6 / 46.0 / 56.8;
//           64 features 157 x 4096 8.0 -> 10.2, 4096 x 4096 16.2 -> 13.1, 16384 x 4096 23.6 -> 43.7
//   g w     4096 x 4096 with 8 / 16 / 32 15.0 / 15.4 / 11.4 -> 10.9 / 11.0 / 10.9, 4096 x 11008 42.9 / 44.2 / 30.7 -> 20.2 / 20.6 / 22.5, 65536 x 2048
//           81.7 / 84.0 / 57.9 -> 52.1 / 58.5 / 68.8, 157 x 4096 5.2 / 5.2 / 4.3 -> 5.8 / 5.8 / 6.1 (the library's call costs the host 20 us more)
int32_t hyc_thin_covers(int64_t M, int64_t K, int64_t N, int32_t input_grad) {
  if (M <= 0 || K <= 0 || N < 8 || N > 32 || N % 8 != 0 || K % 64 != 0 || K > (1 << 24) || M > (int64_t)65535 * LO_M) return 0;
  if (input_grad && N <= 16) return 1;
  return M * K <= (input_grad ? (int64_t)1 << 26 : (int64_t)3 << 24) ? 1 : 0;
}

int hyc_thin_dx(const void* g, int64_t ldg, int64_t M, const void* w, int32_t N, int64_t K, void* dx, void* stream) {
  if (N < 8 || N > 32 || N % 8 != 0) return fail(HYC_ENOTSUP, "hyc_thin_dx: a weight of %d rows (8 to 32, a multiple of 8)", N);
  if (K <= 0 || K % 8 != 0 || K > (1 << 24)) return fail(HYC_ENOTSUP, "hyc_thin_dx: rows of %lld (a multiple of 8)", (long long)K);
  if (M < 0 || ldg < N || ldg % 8 != 0) return fail(HYC_EINVAL, "hyc_thin_dx: M=%lld, row pitch %lld", (long long)M, (long long)ldg);
  if (M == 0) return HYC_OK;
  if (!g || !w || !dx) return fail(HYC_EFAULT, "hyc_thin_dx: null buffer");
  if (!aligned16(g) || !aligned16(dx)) return fail(HYC_EINVAL, "hyc_thin_dx: g and dx must be 16-byte aligned");
  if ((M + LO_M - 1) / LO_M > 65535) return fail(HYC_ENOTSUP, "hyc_thin_dx: too many tokens");
  const dim3 grid((unsigned)((K + LO_F - 1) / LO_F), (unsigned)((M + LO_M - 1) / LO_M));
  hipLaunchKernelGGL(k_thin_dx, grid, dim3(256), 0, begin_launch(stream), static_cast<const uint16_t*>(g), ldg, M,
                     static_cast<const uint16_t*>(w), N, (int)K, static_cast<uint16_t*>(dx));
  return check_launch("hyc_thin_dx");
}

int64_t hyc_lora_up_bwd_workspace_bytes(int64_t M, const int64_t* n_out, int32_t n, int32_t r) {
  if (M <= 0 || !n_out || n < 1 || n > LORA_MAX || r < 1) return 0;
  int64_t rows = 0;
  for (int i = 0; i < n; ++i) rows += n_out[i];
  const int fblocks = lora_up_blocks(n_out, n);
  const int64_t RC = r <= 16 ? 16 : 32;
  return 4 * RC * ((int64_t)fblocks * M + lora_up_ranges(M, fblocks) * rows);
}

int hyc_lora_up_bwd(const void* const* dy, const int64_t* ldg, int64_t M, const int64_t* n_out, const void* const* B, const void* h,
                    int32_t n, int32_t r, float scale, void* dh, void* ext, int64_t ld_ext, int64_t room, int32_t copy_dy, void* const* dB,
                    void* workspace, void* stream) {
  LoraGroup g;
  int rc = lora_group("hyc_lora_up_bwd", B, n_out, n, r, 64, &g);
  if (rc) return rc;
  const int nr = n * r;
  const int64_t rows = g.end[n - 1];
  if (M < 0 || room < nr || room % 8 != 0 || room > 4096 || ld_ext < rows + room || ld_ext % 8 != 0)
    return fail(HYC_EINVAL, "hyc_lora_up_bwd: M=%lld, row pitch %lld, room=%lld for %d columns behind %lld", (long long)M, (long long)ld_ext,
                (long long)room, nr, (long long)rows);
  if (!dy || !ldg || !dB || (M > 0 && (!h || !dh || !ext || !workspace))) return fail(HYC_EFAULT, "hyc_lora_up_bwd: null buffer");
  if (!aligned16(h) || !aligned16(ext) || !aligned16(workspace)) return fail(HYC_EINVAL, "hyc_lora_up_bwd: buffers must be 16-byte aligned");
  LoraUp a = {};
  a.n = n; a.r = r;
  for (int i = 0; i < n; ++i) {
    if ((M > 0 && !dy[i]) || !dB[i]) return fail(HYC_EFAULT, "hyc_lora_up_bwd: null buffer");
    if (!aligned16(dy[i]) || ldg[i] < n_out[i] || ldg[i] % 8 != 0)
      return fail(HYC_EINVAL, "hyc_lora_up_bwd: dy must be 16-byte aligned, rows a multiple of 8 (at least n_out) apart");
    a.g[i] = static_cast<const uint16_t*>(dy[i]);
    a.ldg[i] = ldg[i];
    a.B[i] = g.f[i];
    a.dB[i] = static_cast<uint16_t*>(dB[i]);
    a.n_out[i] = (int)n_out[i];
    a.fb0[i + 1] = a.fb0[i] + (int)((n_out[i] + LU_F - 1) / LU_F);
    a.row0[i + 1] = a.row0[i] + (int)n_out[i];
  }
  const int fblocks = a.fb0[n];
  int64_t pitch = 0;
  for (int i = 0; i < n; ++i) pitch = ldg[i] > pitch ? ldg[i] : pitch;
  const int64_t tokens = lora_up_tokens(M, fblocks, pitch);
  if (tokens * pitch >= LU_RANGE) return fail(HYC_ENOTSUP, "hyc_lora_up_bwd: a token range of dy must stay below 2 GiB");
  const int used = M ? (int)((M + tokens - 1) / tokens) : 0;   // (no tokens: the sums below are empty and dB is zero)
  const int RC = r <= 16 ? 16 : 32;
  float *dhp = static_cast<float*>(workspace), *dbp = dhp + (int64_t)fblocks * M * RC;
  // (the kernel's copy counts 32-bit bytes from one row to the next; rows that far apart are few and go one by one)
  const bool by_rows = copy_dy && ld_ext >= ((int64_t)1 << 29);
  uint16_t* cp = copy_dy && !by_rows ? static_cast<uint16_t*>(ext) : nullptr;
  hipStream_t st = begin_launch(stream);
  for (int i = 0; i < n && by_rows; ++i)
    for (int64_t m = 0; m < M; ++m)
      if (hipMemcpyAsync(static_cast<uint16_t*>(ext) + m * ld_ext + a.row0[i], a.g[i] + m * ldg[i], 2 * (size_t)n_out[i], hipMemcpyDeviceToDevice, st) != hipSuccess)
        return fail(HYC_ELAUNCH, "hyc_lora_up_bwd: a row of dy could not be copied");
  const dim3 grid((unsigned)fblocks, (unsigned)used);
#define HYC_GO(RT_, COPY_)                                                                                                   \
  hipLaunchKernelGGL((k_lora_up_bwd<RT_, COPY_>), grid, dim3(256), 0, st, a, M, static_cast<const uint16_t*>(h), (int)tokens, dhp, dbp, cp, ld_ext)
  if (M > 0) {
    if (RC == 16) { if (cp) HYC_GO(1, true); else HYC_GO(1, false); }
    else { if (cp) HYC_GO(2, true); else HYC_GO(2, false); }
  }
#undef HYC_GO
  if ((rc = check_launch("hyc_lora_up_bwd"))) return rc;
  const int64_t per = 256 / RC, token_blocks = (M + per - 1) / per, blocks = n * token_blocks + (rows + per - 1) / per;
  if (blocks >= ((int64_t)1 << 31)) return fail(HYC_ENOTSUP, "hyc_lora_up_bwd: too many tokens");
#define HYC_GO(RC_)                                                                                                          \
  hipLaunchKernelGGL((k_lora_up_finish<RC_>), dim3((unsigned)blocks), dim3(256), 0, st, a, M, dhp, dbp, used, scale,          \
                     static_cast<uint16_t*>(dh), static_cast<uint16_t*>(ext) + rows, ld_ext, (int)room, (unsigned)token_blocks)
  if (RC == 16) HYC_GO(16);
  else HYC_GO(32);
#undef HYC_GO
  return check_launch("hyc_lora_up_bwd (finish)");
}

}  // extern "C"
