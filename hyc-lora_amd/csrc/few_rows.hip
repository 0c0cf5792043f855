// The products of a LoRA group with its base weight over few tokens, each one launch:
//
//   forward     y = bf16(s h B^T) + x W^T, W decoded from its NF4 codes on the way into the matrix operands
//   backward    dX = ext wt^T, wt as hyc_lora_weight_t writes it
//
// Over a few hundred tokens a product is a walk over the weight, and the library's call costs the host more (20 to 25 us) than the walk
// costs the GPU; the decoded weight, written and read again, is a second launch, and y = s h B^T a third.  What bounds the walk is how
// fast operands reach a CU; with fragments loaded as the matrix operands want them, neighbouring lanes in different rows, 157 tokens x
// 2048 -> 2048 / 6144 / 11264 took 15.7 / 34.5 / 51.1 us instead of 8.2 / 15.9 / 25.5.
#include "abi_util.hpp"
#include "nf4_levels.hpp"

namespace hyc {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
#define HYC_MFMA16(a_, b_, c_) __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_, b_, c_, 0, 0, 0)

constexpr int FR_MAX = 4;                                // projections of a group

struct FewRows {
  const uint16_t* x;                                     // [M, K], rows ldx apart
  int64_t ldx;
  int M, K, N;
  // one of the two weights [N, K]
  const uint8_t* packed;
  const float* absmax;
  const uint16_t* w;                                     // rows K apart
  // the rank-r term (n = 0: none)
  const uint16_t* h;                                     // [M, n r]
  const uint16_t* B[FR_MAX];                             // [n_out_i, r]
  int row0[FR_MAX + 1];
  int n, r;
  float scale;
  uint16_t* y;                                           // [M, N]
};

// A workgroup is WAVES waves on one block of 16 MT tokens x 16 NT features; they deal the reduction out in blocks of 64 and meet in LDS.
// Operands come as whole lines (eight lanes a row of 128 bytes; lanes that go to different rows take the load path several times as
// long) and are turned in LDS of the wave's own, without a barrier; codes are passed on between lanes.  The next block is requested before
// this one is used (the last one twice: a branch around a load would end in a wait).  The features are the rows of the result, so that a
// lane holds four neighbouring ones of a token.
template <int MT, int NT, bool NF4, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, 2)
k_few_rows(FewRows a) {
  constexpr int TILES = MT * NT, WT = NF4 ? 0 : NT;
  constexpr int OWN = (MT + WT) * 1024, RED = WAVES * 512;   // elements of a wave's tiles / of its sums of WAVES tiles (floats as pairs)
  __shared__ __align__(16) uint16_t lds[WAVES][OWN > RED ? OWN : RED];
  __shared__ float lut[16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l15 = lane & 15, lq = lane >> 4;
  if (NF4) {
    if (threadIdx.x < 16) lut[threadIdx.x] = kNF4[threadIdx.x];
    __syncthreads();
  }
  const int n0 = (int)blockIdx.x * 16 * NT, m0 = (int)blockIdx.y * 16 * MT, blocks = a.K / 64;
  const int lr = lane >> 3, lc = lane & 7;               // a load brings eight rows of eight chunks
  uint32_t xo[MT][2], wo[NT][2];                         // byte offsets of this lane's rows (tokens and features past the end repeat the last one)
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int m = m0 + 16 * i + 8 * u + lr;
      xo[i][u] = (uint32_t)(m < a.M ? m : a.M - 1) * (uint32_t)a.ldx * 2u + 16u * lc;
    }
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int u = 0; u < 2; ++u) {                        // (codes: four lanes a row of 32 bytes, one load a tile)
      const int n = n0 + 16 * j + (NF4 ? lane >> 2 : 8 * u + lr);
      wo[j][u] = (uint32_t)(n < a.N ? n : a.N - 1) * (NF4 ? (uint32_t)a.K / 2u : (uint32_t)a.K * 2u) + (NF4 ? 8u * (lane & 3) : 16u * lc);
    }
  const float* absmax[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + 16 * j + l15;
    absmax[j] = NF4 ? a.absmax + (int64_t)(n < a.N ? n : a.N - 1) * blocks : nullptr;
  }
  bf16x8_t xr[MT][2], wr[NF4 ? 1 : NT][2];
  uint2 codes[NF4 ? NT : 1];
  float s_in[NF4 ? NT : 1];
  auto load = [&](int b) __attribute__((always_inline)) {
    const char* xb = reinterpret_cast<const char*>(a.x) + 128 * (int64_t)b;
    const char* wb = NF4 ? reinterpret_cast<const char*>(a.packed) + 32 * (int64_t)b : reinterpret_cast<const char*>(a.w) + 128 * (int64_t)b;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if constexpr (NF4) {
        codes[j] = *reinterpret_cast<const uint2*>(wb + wo[j][0]);
        s_in[j] = absmax[j][b];
      } else {
#pragma unroll
        for (int u = 0; u < 2; ++u) wr[j][u] = *reinterpret_cast<const bf16x8_t*>(wb + wo[j][u]);
      }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int u = 0; u < 2; ++u) xr[i][u] = *reinterpret_cast<const bf16x8_t*>(xb + xo[i][u]);
  };
  floatx4_t acc[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) acc[t] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  uint16_t* T = lds[wave];
  // chunk c of row r lies at c ^ (r / 2 % 8): the 16 lanes of a read and of a write are on all banks
  const int put = lr * 64 + 8 * (lc ^ ((lr >> 1) & 7)), put8 = (8 + lr) * 64 + 8 * (lc ^ (((8 + lr) >> 1) & 7));
  int get[2];                                            // element 8 of a lane's step s: reduction index 16 lq + 8 s of the block
#pragma unroll
  for (int s = 0; s < 2; ++s) get[s] = l15 * 64 + 8 * ((2 * lq + s) ^ ((l15 >> 1) & 7));
  if (wave < blocks) {
    const int last = blocks - 1 - (blocks - 1 - wave) % WAVES;   // this wave's last block
    load(wave);
    for (int b = wave; b < blocks; b += WAVES) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        *reinterpret_cast<bf16x8_t*>(T + i * 1024 + put) = xr[i][0];
        *reinterpret_cast<bf16x8_t*>(T + i * 1024 + put8) = xr[i][1];
      }
      bf16x8_t w[NT][2];
      if constexpr (NF4) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const int from = 4 * l15 + lq;                 // the lane that loaded this row's codes of 16 lq ..
          const uint32_t word[2] = {(uint32_t)__shfl((int)codes[j].x, from, 64), (uint32_t)__shfl((int)codes[j].y, from, 64)};
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            float v[8];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const uint32_t byte = (word[s] >> (8 * q)) & 0xFFu;
              v[2 * q] = lut[byte >> 4] * s_in[j];
              v[2 * q + 1] = lut[byte & 15u] * s_in[j];
            }
            w[j][s] = __builtin_bit_cast(bf16x8_t, pack8(v));
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          *reinterpret_cast<bf16x8_t*>(T + (MT + j) * 1024 + put) = wr[j][0];
          *reinterpret_cast<bf16x8_t*>(T + (MT + j) * 1024 + put8) = wr[j][1];
        }
      }
      load(b + WAVES < last ? b + WAVES : last);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if constexpr (!NF4) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int s = 0; s < 2; ++s) w[j][s] = *reinterpret_cast<const bf16x8_t*>(T + (MT + j) * 1024 + get[s]);
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const bf16x8_t x = *reinterpret_cast<const bf16x8_t*>(T + i * 1024 + get[s]);
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[j * MT + i] = HYC_MFMA16(w[j][s], x, acc[j * MT + i]);
        }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
  // the waves' sums meet in the same memory, WAVES tiles at a time (a wave's own part of it); a wave adds up one tile, in wave order, and writes it
#pragma unroll
  for (int t0 = 0; t0 < TILES; t0 += WAVES) {
    if (t0) __syncthreads();
#pragma unroll
    for (int t = t0; t < t0 + WAVES && t < TILES; ++t) *reinterpret_cast<floatx4_t*>(T + 2 * ((t - t0) * 256 + 4 * lane)) = acc[t];
    __syncthreads();
    const int t = t0 + wave;
    if (t >= TILES) continue;
    floatx4_t sum = *reinterpret_cast<const floatx4_t*>(lds[0] + 2 * (wave * 256 + 4 * lane));
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += *reinterpret_cast<const floatx4_t*>(lds[w] + 2 * (wave * 256 + 4 * lane));
    const int f = n0 + 16 * (t / MT), m = m0 + 16 * (t % MT) + l15;
    if (f >= a.N) continue;                              // (N is a multiple of 16)
    if (NF4 && a.n) {
      int p = 0;
      while (p + 1 < a.n && f >= a.row0[p + 1]) ++p;     // (so are the projections' widths: a tile lies in one of them)
      uint4 vb = make_uint4(0, 0, 0, 0), vh = vb;
      if (8 * lq < a.r) {
        vb = *reinterpret_cast<const uint4*>(a.B[p] + (int64_t)(f - a.row0[p] + l15) * a.r + 8 * lq);
        if (m < a.M) vh = *reinterpret_cast<const uint4*>(a.h + (int64_t)m * (a.n * a.r) + p * a.r + 8 * lq);
      }
      const floatx4_t z = {0.f, 0.f, 0.f, 0.f};
      const floatx4_t up = HYC_MFMA16(__builtin_bit_cast(bf16x8_t, vb), __builtin_bit_cast(bf16x8_t, vh), z);
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[i] += bfr(up[i] * a.scale);   // rounded before it is added, as where it is a tensor of its own
    }
    if (m < a.M) {
      const uint32_t lo = (uint32_t)f_to_bf(sum[0]) | ((uint32_t)f_to_bf(sum[1]) << 16), hi = (uint32_t)f_to_bf(sum[2]) | ((uint32_t)f_to_bf(sum[3]) << 16);
      *reinterpret_cast<uint2*>(a.y + (int64_t)m * a.N + f + 4 * lq) = make_uint2(lo, hi);
    }
  }
}

// Tokens in tiles of up to 4, or of 4 or 5, a workgroup, whichever pads less; features in 1, 2 or 4, the fewest with which the workgroups are resident at
// once, one of eight waves a CU; past that, 4 features' tiles and workgroups of four waves, two a CU (so are those of a weight that goes
// through LDS).
struct FewTiles { int mt, nt, across, down; };           // tiles of a workgroup, workgroups
static FewTiles few_rows_tiles(int64_t M, int64_t N) {
  const int tiles = (int)((M + 15) / 16), across = (int)(N / 16);
  const int mt = tiles <= 4 ? tiles : (tiles + 4) / 5 * 5 < (tiles + 3) / 4 * 4 ? 5 : 4, down = (tiles + mt - 1) / mt;
  // (2048 -> 2048 over 512 tokens with 1 / 2 / 4 tiles of features, us: 17.0 / 14.9 / 13.4; over 256 26.2 in four waves / 9.2 / 12.8)
  const int64_t all = (int64_t)across * down, half = (int64_t)((across + 1) / 2) * down;
  const int nt = all <= 256 ? 1 : half <= 256 ? 2 : 4;
  return {mt, nt, (across + nt - 1) / nt, down};
}
template <bool NF4>
static void few_rows_launch(const FewRows& a, hipStream_t st) {
  const FewTiles t = few_rows_tiles(a.M, a.N);
  const int mt = t.mt, nt = t.nt;
  const dim3 grid((unsigned)t.across, (unsigned)t.down);
  const bool four = nt == 4 && (!NF4 || grid.x * grid.y > 256);
#define HYC_GO(MT_)                                                                                        \
  do {                                                                                                     \
    if (nt == 1) hipLaunchKernelGGL((k_few_rows<MT_, 1, NF4, 8>), grid, dim3(512), 0, st, a);               \
    else if (nt == 2) hipLaunchKernelGGL((k_few_rows<MT_, 2, NF4, 8>), grid, dim3(512), 0, st, a);          \
    else if (four) hipLaunchKernelGGL((k_few_rows<MT_, 4, NF4, 4>), grid, dim3(256), 0, st, a);             \
    else if constexpr (NF4) hipLaunchKernelGGL((k_few_rows<MT_, 4, NF4, 8>), grid, dim3(512), 0, st, a);    \
  } while (0)
  switch (mt) {
    case 1: HYC_GO(1); break;
    case 2: HYC_GO(2); break;
    case 3: HYC_GO(3); break;
    case 4: HYC_GO(4); break;
    default: HYC_GO(5); break;
  }
#undef HYC_GO
}

}  // namespace hyc

using namespace hyc;

extern "C" {

// Where these products are taken.  GPU time, us, library with its decoding and k_lora_up (forward) or alone (dX) -> one launch here; a
// library call costs the host 21 to 30 us beside it, one of these 5.
//   forward K -> N      16 tokens      157            256            512            1024           2048
//   1024 -> 1024        11.8 -> 3.5    16.6 -> 5.5    17.5 -> 5.2    18.0 -> 6.7    19.2 -> 9.5    21.8 -> 14.9
//   1024 -> 5632        17.2 -> 4.5    25.3 -> 11.2   28.6 -> 14.3   32.9 -> 22.0   41.5 -> 37.1   54.7 -> 64.8
//   2048 -> 2048        17.2 -> 4.4    21.1 -> 8.2    25.2 -> 9.5    27.4 -> 13.3   31.4 -> 22.9   37.1 -> 41.7
//   2048 -> 6144        29.0 -> 6.3    37.1 -> 15.9   40.0 -> 22.8   38.9 -> 33.2   46.7 -> 58.7
//   2048 -> 11264       27.8 -> 11.5   39.4 -> 25.5   43.3 -> 32.9   52.2 -> 57.7   75.3 -> 102
//   5632 -> 2048        24.6 -> 7.3    33.9 -> 17.0   32.8 -> 19.1   34.1 -> 27.7   47.7 -> 49.5
//   4096 -> 12288       45.4 -> 19.9   58.9 -> 42.9   69.2 -> 56.6   80.0 -> 104
//   11008 -> 4096       49.2 -> 15.5   59.4 -> 36.4   61.8 -> 48.0   86.7 -> 90.5
//   dX N -> K           16             157            256            512            1024           2048
//   1024 -> 1024        5.5 -> 2.8     5.5 -> 4.8     5.6 -> 4.7     6.6 -> 5.7     7.9 -> 7.6     10.4 -> 12.3
//   3072 -> 1024        10.0 -> 4.0    10.7 -> 8.3    13.5 -> 7.7    16.3 -> 9.7    19.2 -> 13.9   21.7 -> 24.4
//   2048 -> 2048        8.7 -> 3.5     9.6 -> 7.1     13.5 -> 7.4    14.1 -> 10.7   16.0 -> 17.1   22.0 -> 30.8
//   11264 -> 2048       30.5 -> 11.4   37.0 -> 25.4   38.4 -> 25.7   46.7 -> 37.9   66.6 -> 67.2
//   2048 -> 5632        11.2 -> 5.9    14.6 -> 11.8   19.4 -> 16.5   19.4 -> 23.8   29.2 -> 42.5
//   12288 -> 4096       33.4 -> 16.7   46.8 -> 35.5   49.5 -> 40.8   71.1 -> 75.8
//   4096 -> 11008       27.2 -> 16.7   30.5 -> 38.7   38.9 -> 54.6
// A workgroup's tiles share their operands with no other one, so what a launch reads grows with the products of the sides.  dX is
// better, whatever the reduction, while its workgroups are resident at once, one a CU, and its result has at most 2^20 elements.  One
// more block of tokens is a second round, us, library -> here, just below | just above:
//   N 11008, K 4160     80 tokens 27.1 -> 19.0 | 81 26.2 -> 34.2, 95 26.4 -> 34.7
//   N 5632, K 2112      160       15.6 -> 11.6 | 161 15.0 -> 15.7, 186 15.1 -> 15.8
//   N 2816, K 1088      320       7.9 -> 7.7   | 321 8.9 -> 10.0, 350 8.8 -> 10.2
//   N 1536, K 4160                             | 680 25.0 -> 25.9
// A single block of tokens pays past that too (N 22016, K 4160: 16 tokens 67.7 -> 38.4, 40 45.8 -> 45.2; 32768: 16 60.0 -> 46.8, 32 50.8
// -> 48.9): every weight row is read by one workgroup.
// The forward, which saves a pass over the decoded weight as well, is taken up to 256 tokens, whatever the weight, and beyond them until
// about 6e9 multiplications.  From 193 tokens on the library comes level at a few widths: 4096 -> 22016 over 157 / 192 / 224 / 256 tokens
// 89.2 -> 65.9 / 95.6 -> 87.1 / 97.9 -> 97.3 / 101.5 -> 102.5, 5120 -> 15360 over 224 / 241 / 256 94.8 -> 79.2 / 84.9 -> 90.5 / 95.1 -> 88.4, 3072 ->
// 16384 over 241 62.0 -> 63.0; beside them 4096 -> 28672 over 256 148 -> 127, 5120 -> 27648 180 -> 155, 13824 -> 5120 138 -> 107, 8192 ->
// 57344 over 16 / 157 / 256 479 -> 133 / 508 -> 303 / 518 -> 516, 28672 -> 8192 over 256 453 -> 247.
int32_t hyc_few_rows_covers(int64_t M, int64_t K, int64_t N, int32_t input_grad) {
  if (M <= 0 || K <= 0 || N <= 0 || K % 64 != 0 || N % 16 != 0 || K > (1 << 24) || N > (1 << 24)) return 0;
  if (M * K >= ((int64_t)1 << 30) || N * K >= ((int64_t)1 << 30)) return 0;
  if (input_grad) {
    if (M > 1024 || M * N > (1 << 20)) return 0;
    const FewTiles t = few_rows_tiles(M, N);
    return t.down == 1 || (int64_t)t.across * t.down <= 256 ? 1 : 0;
  }
  return M <= 256 || (M <= 2048 && M * K * N <= (int64_t)6000000000) ? 1 : 0;
}

static int few_rows_args(const char* who, const void* x, int64_t ldx, int64_t M, int64_t K, int64_t N, const void* w, const void* y) {
  if (M < 0 || M > 16 * 65535 || K <= 0 || K % 64 != 0 || K > (1 << 24) || N <= 0 || N % 16 != 0 || N > (1 << 24))
    return fail(HYC_ENOTSUP, "%s: [%lld, %lld] x [%lld, %lld]^T (K a multiple of 64, N of 16)", who, (long long)M, (long long)K, (long long)N, (long long)K);
  if (ldx < K || ldx % 8 != 0) return fail(HYC_EINVAL, "%s: row pitch %lld", who, (long long)ldx);
  if (M * ldx >= ((int64_t)1 << 30) || N * K >= ((int64_t)1 << 30)) return fail(HYC_ENOTSUP, "%s: an operand must stay below 2 GiB", who);
  if (M == 0) return HYC_OK;
  if (!x || !w || !y) return fail(HYC_EFAULT, "%s: null buffer", who);
  if (!aligned16(x) || !aligned16(w) || !aligned16(y)) return fail(HYC_EINVAL, "%s: buffers must be 16-byte aligned", who);
  return HYC_OK;
}

int hyc_few_rows_nf4(const void* x, int64_t ldx, int64_t M, int64_t K, const void* packed, const float* absmax, const void* h, const void* const* B,
                     const int64_t* n_out, int32_t n, int32_t r, float scale, void* y, void* stream) {
  if (n < 1 || n > FR_MAX) return fail(HYC_ENOTSUP, "hyc_few_rows_nf4: %d projections (1 to %d)", n, FR_MAX);
  if (r < 8 || r > 32 || r % 8 != 0) return fail(HYC_ENOTSUP, "hyc_few_rows_nf4: rank %d (8, 16, 24 or 32)", r);
  if (!B || !n_out) return fail(HYC_EFAULT, "hyc_few_rows_nf4: null buffer");
  FewRows a = {};
  int64_t N = 0;
  for (int i = 0; i < n; ++i) {
    if (!B[i]) return fail(HYC_EFAULT, "hyc_few_rows_nf4: null factor");
    if (!aligned16(B[i])) return fail(HYC_EINVAL, "hyc_few_rows_nf4: factors must be 16-byte aligned");
    if (n_out[i] <= 0 || n_out[i] % 16 != 0 || n_out[i] > (1 << 24)) return fail(HYC_ENOTSUP, "hyc_few_rows_nf4: %lld output features (a multiple of 16)", (long long)n_out[i]);
    a.B[i] = static_cast<const uint16_t*>(B[i]);
    a.row0[i] = (int)N;
    N += n_out[i];
  }
  for (int i = n; i <= FR_MAX; ++i) a.row0[i] = (int)N;
  int rc = few_rows_args("hyc_few_rows_nf4", x, ldx, M, K, N, packed, y);
  if (rc || M == 0) return rc;
  if (!h || !absmax) return fail(HYC_EFAULT, "hyc_few_rows_nf4: null buffer");
  if (!aligned16(h)) return fail(HYC_EINVAL, "hyc_few_rows_nf4: buffers must be 16-byte aligned");
  a.x = static_cast<const uint16_t*>(x); a.ldx = ldx; a.M = (int)M; a.K = (int)K; a.N = (int)N;
  a.packed = static_cast<const uint8_t*>(packed); a.absmax = absmax;
  a.h = static_cast<const uint16_t*>(h); a.n = n; a.r = r; a.scale = scale;
  a.y = static_cast<uint16_t*>(y);
  few_rows_launch<true>(a, begin_launch(stream));
  return check_launch("hyc_few_rows_nf4");
}

int hyc_few_rows(const void* x, int64_t ldx, int64_t M, int64_t K, const void* w, int64_t N, void* y, void* stream) {
  int rc = few_rows_args("hyc_few_rows", x, ldx, M, K, N, w, y);
  if (rc || M == 0) return rc;
  FewRows a = {};
  a.x = static_cast<const uint16_t*>(x); a.ldx = ldx; a.M = (int)M; a.K = (int)K; a.N = (int)N;
  a.w = static_cast<const uint16_t*>(w);
  a.y = static_cast<uint16_t*>(y);
  few_rows_launch<false>(a, begin_launch(stream));
  return check_launch("hyc_few_rows");
}

}  // extern "C"
