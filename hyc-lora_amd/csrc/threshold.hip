// The threshold scheme's two hot passes for rows of one 8-channel chunk per thread and segment, 4- or 8-bit codes and a base of rank
// 0 to 2: x -> codes, per-row counts and the kept elements in a slab, alone or with the RMSNorm / LayerNorm of the same read
// (operators/compress_function.py:136-200 with efficient_rmsnorm.py:15-60, efficient_layernorm.py:15-61), and codes + CSR -> x_hat
// (compress_function.py:203-261).
//
// The general kernels (norm.hip, compress.hip) are bound by their vector instructions, not by memory: a division per element where
// the scale is per channel, and the base's rows and the scales loaded and unpacked for every row.  Scale, reciprocal, base and
// weight columns belong to a channel, and a thread owns the same channels of every row it walks, so they are held in
// registers here; and the kept elements leave while the row is there (as softmax.hip's slab) instead of in a second read of x.
// 4 x 1024 x 4096, 8-bit codes per channel, rank 2, us (kernel trace): RMSNorm + codes 35 -> 26, kept elements 16 -> 4, x_hat 18 -> 16;
// 16 384 rows: 89, 6 and 52 (3.8, and 4.0 TB/s).  What is left is the chain of a row - loads, two sums, a barrier, stores - with two
// workgroups of eight waves on a CU (103 registers).  These kernels hold everything for 4- and 8-bit codes; 1- and 2-bit codes would
// take four and eight chunks' constants per thread, and keep the general kernels.
#include "abi_util.hpp"
#include "row_kernels.hpp"
#include "threshold.hpp"
#include "wave_scan.hpp"

namespace hyc {

__device__ __forceinline__ void load_vec8(const void* p, bool f32, int64_t col, float (&o)[8]) {
  if (f32) {
    const float4 a = *reinterpret_cast<const float4*>(static_cast<const float*>(p) + col);
    const float4 b = *reinterpret_cast<const float4*>(static_cast<const float*>(p) + col + 4);
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
  } else {
    unpack8(*reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p) + col), o);
  }
}

// codes8 with a scale per element, r = 1 / s of scales within (1e-30, 1e30) (see Recip); s: for the IEEE division otherwise
template <int BITS>
__device__ __forceinline__ void codes8_per_channel(const float (&v)[8], const float (&r)[8], const uint4& s, bool plain, uint32_t& lo, uint32_t& hi) {
  constexpr float MAGIC = 12582912.0f + (BITS == 8 ? 0.f : (float)Q<BITS>::OFF);
  uint32_t u[8];
  if (__builtin_expect(plain, 1)) {
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const uint32_t pk = pack_bf16(v[j] * r[j], v[j + 1] * r[j + 1]);
      u[j] = __float_as_uint(__builtin_amdgcn_fmed3f(bf_lo(pk), Q<BITS>::LO, Q<BITS>::HI) + MAGIC);
      u[j + 1] = __float_as_uint(__builtin_amdgcn_fmed3f(bf_hi(pk), Q<BITS>::LO, Q<BITS>::HI) + MAGIC);
    }
  } else {
    float sv[8];
    unpack8(s, sv);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float t = __builtin_rintf(bfr(v[j] / sv[j]));
      t = (t != t) ? 0.f : t;
      u[j] = __float_as_uint(__builtin_fminf(__builtin_fmaxf(t, Q<BITS>::LO), Q<BITS>::HI) + MAGIC);
    }
  }
  const uint32_t p01 = __builtin_amdgcn_perm(u[1], u[0], 0x0c0c0400u), p23 = __builtin_amdgcn_perm(u[3], u[2], 0x0c0c0400u);
  const uint32_t p45 = __builtin_amdgcn_perm(u[5], u[4], 0x0c0c0400u), p67 = __builtin_amdgcn_perm(u[7], u[6], 0x0c0c0400u);
  lo = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
  hi = __builtin_amdgcn_perm(p67, p45, 0x05040100u);
}

// the base of rank up to 2 at one chunk of channels: its two rows as packed bf16 (a second row of zeros for rank 1)
struct Base2 {
  uint4 r0, r1;
  __device__ __forceinline__ void load(const ThrArgs& a, int64_t col, int64_t H) {
    r0 = *reinterpret_cast<const uint4*>(a.R + col);
    r1 = a.rank > 1 ? *reinterpret_cast<const uint4*>(a.R + H + col) : make_uint4(0, 0, 0, 0);
  }
  __device__ __forceinline__ void at(float l0, float l1, float (&b)[8]) const {
    float x[8], y[8];
    unpack8(r0, x);
    unpack8(r1, y);
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const uint32_t pk = pack_bf16(__builtin_fmaf(l1, y[j], __builtin_fmaf(l0, x[j], 0.f)), __builtin_fmaf(l1, y[j + 1], __builtin_fmaf(l0, x[j + 1], 0.f)));
      b[j] = bf_lo(pk);
      b[j + 1] = bf_hi(pk);
    }
  }
};
__device__ __forceinline__ void base_row(const ThrArgs& a, int pos, float& l0, float& l1) {
  l0 = bf_to_f(a.L[(int64_t)pos * a.rank]);
  l1 = a.rank > 1 ? bf_to_f(a.L[(int64_t)pos * a.rank + 1]) : 0.f;
}

// NORM: 0 compress only, 1 RMSNorm, 2 LayerNorm.  One row per workgroup and iteration, the next one requested ahead; sums and counts
// of a row meet in LDS behind one barrier (two for LayerNorm).
template <int BITS, int NORM, bool PERCHAN, bool BASE, int MAXT>
__global__ void __launch_bounds__(MAXT)
k_thr_fwd(const uint16_t* __restrict__ x, const void* __restrict__ w, const void* __restrict__ bias, bool wf32, float eps, int64_t M, int64_t H,
          int CPS, ThrArgs a, uint16_t* __restrict__ y, float* __restrict__ mean_out, float* __restrict__ rstd_out, uint8_t* __restrict__ stored,
          int32_t* __restrict__ counts, uint32_t* __restrict__ slab, int cap) {
  constexpr int NSEG = Q<BITS>::NSEG;
  static_assert(NSEG <= 2, "two counts share a word");
  __shared__ float red[2][16];
  __shared__ int cnt[2][16];
  const int64_t SEG = (int64_t)CPS * 8;
  const float invH = 1.0f / (float)H;
  const int wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6, c = threadIdx.x;
  const bool act = c < CPS;
  const int cc = act ? c : 0;                                           // (an idle lane reads chunk 0 of the constants)
  float rec[PERCHAN ? NSEG : 1][8], wv[NORM ? NSEG : 1][8], bv[NORM == 2 ? NSEG : 1][8];
  uint4 sc[PERCHAN ? NSEG : 1];
  Base2 base[BASE ? NSEG : 1];
  bool plain = true;
#pragma unroll
  for (int i = 0; i < NSEG; ++i) {
    const int64_t col = i * SEG + 8 * cc;
    if (PERCHAN) {
      sc[i] = *reinterpret_cast<const uint4*>(a.scale + col);
      unpack8(sc[i], rec[i]);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        plain = plain && rec[i][j] > 1e-30f && rec[i][j] < 1e30f;
        rec[i][j] = 1.0f / rec[i][j];
      }
    }
    if (BASE) base[i].load(a, col, H);
    if (NORM) load_vec8(w, wf32, col, wv[i]);
    if (NORM == 2) {
#pragma unroll
      for (int j = 0; j < 8; ++j) bv[i][j] = 0.f;
      if (bias) load_vec8(bias, wf32, col, bv[i]);
    }
  }
  plain = __ballot(!plain) == 0;
  const int S = (int)a.S, step = (int)(gridDim.x % (unsigned)S);
  int pos = (int)(blockIdx.x % (unsigned)S);
  uint4 raw[NSEG];
  int64_t row = blockIdx.x;
#pragma unroll
  for (int i = 0; i < NSEG; ++i) raw[i] = act && row < M ? *reinterpret_cast<const uint4*>(x + row * H + i * SEG + 8 * c) : make_uint4(0, 0, 0, 0);
  int parity = 0;
  for (; row < M; row += gridDim.x, parity ^= 1) {
    uint4 nxt[NSEG];
    const int64_t nrow = row + gridDim.x;
#pragma unroll
    for (int i = 0; i < NSEG; ++i) nxt[i] = act && nrow < M ? *reinterpret_cast<const uint4*>(x + nrow * H + i * SEG + 8 * c) : make_uint4(0, 0, 0, 0);
    float l0 = 0.f, l1 = 0.f, s_row = 0.f;
    if (BASE) base_row(a, pos, l0, l1);
    if (!PERCHAN) s_row = bf_to_f(a.scale[(int64_t)pos * a.sst]);
    pos += step;
    pos = pos >= S ? pos - S : pos;
    float ss = 0.f;
    uint32_t lo = 0, hi = 0, hot[NSEG];
    uint4 kept[NSEG];                                                   // the elements without the base
#pragma unroll
    for (int i = 0; i < NSEG; ++i) {
      float v[8];
      unpack8(raw[i], v);
      if (NORM) {
#pragma unroll
        for (int j = 0; j < 8; ++j) ss = NORM == 2 ? ss + v[j] : __builtin_fmaf(v[j], v[j], ss);
      }
      kept[i] = raw[i];
      if (BASE) {
        float b[8];
        base[i].at(l0, l1, b);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] -= b[j];
        kept[i] = pack8(v);
        unpack8(kept[i], v);
      }
      hot[i] = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool h = __builtin_fabsf(v[j]) > a.thr;
        hot[i] |= h ? 1u << j : 0u;
        v[j] = h ? 0.f : v[j];
      }
      if (!act) hot[i] = 0;
      uint32_t cl, ch;
      if (PERCHAN) codes8_per_channel<BITS>(v, rec[i], sc[i], plain, cl, ch);
      else codes8<BITS>(v, s_row, cl, ch);
      if (BITS == 8) { lo = cl; hi = ch; }
      else { lo |= cl << (i * BITS); hi |= ch << (i * BITS); }
    }
    if (act) *reinterpret_cast<uint2*>(stored + row * SEG + 8 * c) = make_uint2(lo, hi);
    // kept elements of the row in column order: segment by segment, the two segments' counts in one word
    const int mine = __popc(hot[0]) | (NSEG > 1 ? __popc(hot[NSEG - 1]) << 16 : 0);
    const int incl = wave_inclusive_scan(mine), all = __builtin_amdgcn_readlane(incl, 63);
    if (NORM) ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) {
      if (NORM) red[parity][wave] = ss;
      cnt[parity][wave] = all;
    }
    __syncthreads();
    float sum = 0.f;
    int before = 0, total = 0;
    for (int k = 0; k < nw; ++k) {
      if (NORM) sum += red[parity][k];
      const int n = cnt[parity][k];
      total += n;
      before += k < wave ? n : 0;
    }
    const int at = before + incl - mine, first = total & 0xFFFF;
    uint32_t* srow = slab + row * cap;
#pragma unroll
    for (int i = 0; i < NSEG; ++i) {
      int p = i ? first + (int)((uint32_t)at >> 16) : at & 0xFFFF;
      for (uint32_t m = hot[i]; m; m &= m - 1, ++p) {                    // (about one element in a hundred)
        const int j = __builtin_ctz(m);
        const uint32_t lo2 = j & 2 ? kept[i].y : kept[i].x, hi2 = j & 2 ? kept[i].w : kept[i].z, two = j & 4 ? hi2 : lo2;
        if (p < cap) srow[p] = (uint32_t)(i * SEG + 8 * c + j) | ((j & 1 ? two >> 16 : two & 0xFFFFu) << 16);
      }
    }
    float mean = 0.f;
    if (NORM == 2) {
      mean = sum * invH;
      float var = 0.f;
      if (act) {
#pragma unroll
        for (int i = 0; i < NSEG; ++i) {
          float v[8];
          unpack8(raw[i], v);
#pragma unroll
          for (int j = 0; j < 8; ++j) { const float dlt = v[j] - mean; var = __builtin_fmaf(dlt, dlt, var); }
        }
      }
      parity ^= 1;
      var = wave_sum(var);
      if ((threadIdx.x & 63) == 0) red[parity][wave] = var;
      __syncthreads();
      sum = 0.f;
      for (int k = 0; k < nw; ++k) sum += red[parity][k];
    }
    const float rstd = NORM ? 1.0f / __builtin_sqrtf(sum * invH + eps) : 0.f;
    if (threadIdx.x == 0) {
      counts[row] = first + (int)((uint32_t)total >> 16);
      if (NORM) rstd_out[row] = rstd;
      if (NORM == 2) mean_out[row] = mean;
    }
    if (NORM && act) {
#pragma unroll
      for (int i = 0; i < NSEG; ++i) {
        float v[8];
        unpack8(raw[i], v);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = NORM == 2 ? ((v[j] - mean) * rstd) * wv[i][j] + bv[i][j] : (v[j] * rstd) * wv[i][j];
        store_stream(y + row * H + i * SEG + 8 * c, pack8(v));
      }
    }
#pragma unroll
    for (int i = 0; i < NSEG; ++i) raw[i] = nxt[i];
  }
}

// x_hat = bf16(bf16(base + outlier) + dequant).  The row is put together in LDS (double-buffered: two barriers a row): chunks by their
// threads, then the CSR entries by whichever thread holds one; the codes wait there too for the entries' own dequant (0 unless the
// caller's entries are not the ones that were left out).
template <int BITS, bool PERCHAN, bool BASE, int MAXT>
__global__ void __launch_bounds__(MAXT)
k_thr_restore(const uint8_t* __restrict__ stored, int64_t M, int64_t H, int CPS, ThrArgs a, uint16_t* __restrict__ xhat) {
  constexpr int NSEG = Q<BITS>::NSEG;
  constexpr float OFFV = BITS == 8 ? 128.f : (float)Q<BITS>::OFF;
  extern __shared__ __align__(16) uint16_t rows[];                      // [2][H] values, then [2][CPS] code words
  const int64_t SEG = (int64_t)CPS * 8;
  uint2* words = reinterpret_cast<uint2*>(rows + 2 * H);
  const int c = threadIdx.x;
  const bool act = c < CPS;
  const int cc = act ? c : 0;
  float sv[PERCHAN ? NSEG : 1][8];
  Base2 base[BASE ? NSEG : 1];
#pragma unroll
  for (int i = 0; i < NSEG; ++i) {
    const int64_t col = i * SEG + 8 * cc;
    if (PERCHAN) unpack8(*reinterpret_cast<const uint4*>(a.scale + col), sv[i]);
    if (BASE) base[i].load(a, col, H);
  }
  const int S = (int)a.S, step = (int)(gridDim.x % (unsigned)S);
  int pos = (int)(blockIdx.x % (unsigned)S);
  int64_t row = blockIdx.x;
  uint2 word = make_uint2(0, 0);
  int e0 = 0, e1 = 0, col0 = 0;
  uint32_t val0 = 0;
  auto request = [&](int64_t r) __attribute__((always_inline)) {
    word = act ? *reinterpret_cast<const uint2*>(stored + r * SEG + 8 * c) : make_uint2(0, 0);
    e0 = a.row_ptr[r];
    e1 = a.row_ptr[r + 1];
    if (e0 + c < e1) { col0 = a.cols[e0 + c]; val0 = a.vals[e0 + c]; }
  };
  if (row < M) request(row);
  for (int parity = 0; row < M; row += gridDim.x, parity ^= 1) {
    uint16_t* buf = rows + parity * H;
    uint2* wbuf = words + parity * CPS;
    float l0 = 0.f, l1 = 0.f, s_row = 0.f;
    if (BASE) base_row(a, pos, l0, l1);
    if (!PERCHAN) s_row = bf_to_f(a.scale[(int64_t)pos * a.sst]);
    pos += step;
    pos = pos >= S ? pos - S : pos;
    if (act) {
      wbuf[c] = word;
#pragma unroll
      for (int i = 0; i < NSEG; ++i) {
        constexpr uint32_t REP = BITS == 8 ? 0x80808080u : Q<BITS>::CODE_MASK * 0x01010101u;
        uint32_t p = BITS == 8 ? word.x ^ REP : (word.x >> (i * BITS)) & REP, q = BITS == 8 ? word.y ^ REP : (word.y >> (i * BITS)) & REP;
        asm volatile("" : "+v"(p), "+v"(q));                            // see dequant8
        float f[8];
        codes8_to_float<BITS>(p, q, f);
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] = (f[j] - OFFV) * (PERCHAN ? sv[i][j] : s_row);
        if (BASE) {
          float b[8], d[8];
          base[i].at(l0, l1, b);
          unpack8(pack8(f), d);
#pragma unroll
          for (int j = 0; j < 8; ++j) f[j] = (b[j] + 0.f) + d[j];
        } else {
          float d[8];
          unpack8(pack8(f), d);
#pragma unroll
          for (int j = 0; j < 8; ++j) f[j] = 0.f + d[j];
        }
        *reinterpret_cast<uint4*>(buf + i * SEG + 8 * c) = pack8(f);
      }
    }
    __syncthreads();
    auto place = [&](int col, uint32_t val) __attribute__((always_inline)) {
      const int i = NSEG > 1 && col >= (int)SEG ? 1 : 0, k = col - i * (int)SEG;
      const uint32_t byte = reinterpret_cast<const uint8_t*>(wbuf)[k];
      const float q = BITS == 8 ? (float)(int)(int8_t)byte : (float)((int)((byte >> (i * BITS)) & Q<BITS>::CODE_MASK) - Q<BITS>::OFF);
      const float s = PERCHAN ? bf_to_f(a.scale[col]) : s_row;
      float b = 0.f;
      if (BASE) {
        b = __builtin_fmaf(l0, bf_to_f(a.R[col]), 0.f);
        if (a.rank > 1) b = __builtin_fmaf(l1, bf_to_f(a.R[H + col]), b);
        b = bfr(b);
      }
      buf[col] = f_to_bf(bfr(b + bf_to_f((uint16_t)val)) + bfr(q * s));
    };
    if (e0 + c < e1) place(col0, val0);
    for (int e = e0 + c + (int)blockDim.x; e < e1; e += blockDim.x) place(a.cols[e], a.vals[e]);
    const int64_t nrow = row + gridDim.x;
    if (nrow < M) request(nrow);
    __syncthreads();
    if (act) {
#pragma unroll
      for (int i = 0; i < NSEG; ++i)
        store_stream(xhat + row * H + i * SEG + 8 * c, *reinterpret_cast<const uint4*>(buf + i * SEG + 8 * c));
    }
  }
}

// what both kernels cover: 4- and 8-bit codes, rows of at most 1024 chunks per segment, rank up to 2, a scale that depends on the
// channel or on the row but not on both
static bool covered(const RowGeom& g, const ThrArgs& a, bool perchan, int64_t M) {
  return (g.bits == 4 || g.bits == 8) && g.cps <= 1024 && a.rank <= 2 && (!perchan || a.sst == 0) && a.S < ((int64_t)1 << 31) && M < ((int64_t)1 << 31);
}

// workgroups: `waves` per CU in one round, so that the constants a thread loads serve many rows
static int thr_grid(int64_t M, int threads, int waves) {
  const int64_t g = (int64_t)256 * waves * 64 / threads;
  return (int)(M < g ? M : g);
}

bool launch_thr_restore(const void* stored, int64_t M, int64_t H, const RowGeom& g, const ThrArgs& a, bool perchan, void* xhat, hipStream_t st) {
  const size_t lds = (size_t)4 * H + (size_t)16 * g.cps;
  if (!covered(g, a, perchan, M) || lds > 64 * 1024) return false;
  const int T = g.threads, grid = thr_grid(M, T, 32);
#define HYC_TR(B_, P_, R_)                                                                                                                 \
  do {                                                                                                                                     \
    if (T <= 256) hipLaunchKernelGGL((k_thr_restore<B_, P_, R_, 256>), dim3(grid), dim3(T), lds, st, (const uint8_t*)stored, M, H, g.cps, a, \
                                     (uint16_t*)xhat);                                                                                     \
    else hipLaunchKernelGGL((k_thr_restore<B_, P_, R_, 1024>), dim3(grid), dim3(T), lds, st, (const uint8_t*)stored, M, H, g.cps, a,          \
                            (uint16_t*)xhat);                                                                                              \
  } while (0)
#define HYC_TR_B(B_)                                                                                  \
  do {                                                                                                \
    if (perchan) { if (a.rank) HYC_TR(B_, true, true); else HYC_TR(B_, true, false); }                \
    else { if (a.rank) HYC_TR(B_, false, true); else HYC_TR(B_, false, false); }                      \
  } while (0)
  if (g.bits == 4) HYC_TR_B(4);
  else HYC_TR_B(8);
#undef HYC_TR_B
#undef HYC_TR
  return true;
}

}  // namespace hyc

using namespace hyc;

extern "C" {

int hyc_threshold_fwd(int32_t norm, const void* x, const void* w, const void* bias, int32_t w_dtype, float eps, int64_t M, int64_t H,
                      const hyc_desc* d, void* y, float* mean, float* rstd, void* stored, int32_t* counts, uint32_t* slab, int64_t cap, void* stream) {
  if (!d) return fail(HYC_EFAULT, "hyc_threshold_fwd: null descriptor");
  if (norm < 0 || norm > 2) return fail(HYC_EINVAL, "hyc_threshold_fwd: norm=%d", norm);
  if (M < 0) return fail(HYC_EINVAL, "hyc_threshold_fwd: M=%lld", (long long)M);
  if (d->mode != HYC_MODE_THRESHOLD) return fail(HYC_EINVAL, "hyc_threshold_fwd: threshold mode only");
  if (norm && w_dtype != HYC_DTYPE_BF16 && w_dtype != HYC_DTYPE_F32) return fail(HYC_EINVAL, "hyc_threshold_fwd: w_dtype=%d", w_dtype);
  RowGeom g;
  ThrArgs a;
  bool perchan;
  int rc = row_geom(H, d->bits, &g);
  if (!rc) rc = make_thr_args(d, g, &a, &perchan);
  if (rc) return rc;
  if (!covered(g, a, perchan, M))
    return fail(HYC_ENOTSUP, "hyc_threshold_fwd: H=%lld bits=%d rank=%d (4- or 8-bit codes, H*bits/64 <= 1024, rank <= 2)", (long long)H, d->bits, a.rank);
  if (cap <= 0 || cap > H) return fail(HYC_EINVAL, "hyc_threshold_fwd: cap=%lld must be in 1..H=%lld", (long long)cap, (long long)H);
  if (M == 0) return HYC_OK;
  if (!x || !stored || !counts || !slab || (norm && (!w || !y || !rstd)) || (norm == 2 && !mean)) return fail(HYC_EFAULT, "hyc_threshold_fwd: null buffer");
  if (!aligned16(x) || !aligned8(stored) || (norm && (!aligned16(w) || !aligned16(y))) || (norm == 2 && bias && !aligned16(bias)))
    return fail(HYC_EINVAL, "hyc_threshold_fwd: x, y, w, bias must be 16-byte and stored 8-byte aligned");
  hipStream_t st = begin_launch(stream);
  const int T = g.threads, grid = thr_grid(M, T, 16);
  const bool wf32 = w_dtype == HYC_DTYPE_F32;
#define HYC_TF_K(B_, N_, P_, R_, MT_)                                                                                                       \
  hipLaunchKernelGGL((k_thr_fwd<B_, N_, P_, R_, MT_>), dim3(grid), dim3(T), 0, st, (const uint16_t*)x, w, bias, wf32, eps, M, H, g.cps, a,     \
                     (uint16_t*)y, mean, rstd, (uint8_t*)stored, counts, slab, (int)cap)
#define HYC_TF_R(B_, N_, P_, R_) do { if (T <= 256) HYC_TF_K(B_, N_, P_, R_, 256); else HYC_TF_K(B_, N_, P_, R_, 1024); } while (0)
#define HYC_TF_P(B_, N_)                                                                                    \
  do {                                                                                                      \
    if (perchan) { if (a.rank) HYC_TF_R(B_, N_, true, true); else HYC_TF_R(B_, N_, true, false); }          \
    else { if (a.rank) HYC_TF_R(B_, N_, false, true); else HYC_TF_R(B_, N_, false, false); }                \
  } while (0)
#define HYC_TF(B_) do { if (norm == 0) HYC_TF_P(B_, 0); else if (norm == 1) HYC_TF_P(B_, 1); else HYC_TF_P(B_, 2); } while (0)
  if (d->bits == 4) HYC_TF(4);
  else HYC_TF(8);
#undef HYC_TF
#undef HYC_TF_P
#undef HYC_TF_R
#undef HYC_TF_K
  return check_launch("hyc_threshold_fwd");
}

}  // extern "C"
