// The saved activations of fused attention, all of a pass in one launch each way: forward, q and k through the rotary embedding
// (rope.hip's arithmetic) and q, k and v into codes (compress.hip's); backward, q, k and v out of them and, where the attention's
// output is kept too, the row terms of the gradient from its codes (k_attn_delta's sums), which is never written out.
#include "abi_util.hpp"
#include "row_kernels.hpp"

namespace hyc {

// value of the lane HD / 16 away inside the HD / 8 lanes that hold a head: its other half
template <int HD>
__device__ __forceinline__ uint32_t other_half(uint32_t v) {
  if (HD == 128) return __builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, false);                  // row_ror:8
  v = __builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, false);                                    // row_half_mirror, and each quad
  return __builtin_amdgcn_mov_dpp((int)v, 0x1B, 0xF, 0xF, false);                                  // turned round again
}

struct SiteIn {
  const uint16_t* x;                                     // rows ldx apart
  int64_t ldx;
  uint16_t* rows;                                        // the rotated rows, contiguous; null: not rotated
  uint8_t* stored;
  uint16_t *vals, *scales;
  ChanArgs a;
};
struct SiteIns { SiteIn t[3]; };

// k_compress_chan_fast for three tensors (blockIdx.y), two of them rotated on the way.  A lane's chunk and the chunk of the other half of
// its head are HD / 16 lanes apart, so the rotation is two or four DPP moves a word; outlier channels are rotated once more by
// the lanes that gather them.  Bound by memory: two reads of a matrix less than rotation and compression by themselves.  In a layer
// of 4 x 1024 x 32 x 128, 4 bits: five launches of 50 us -> one of 34 (193 MB, 5.6 TB/s); 157 x 16 x 128, 8 bits: 16.5 -> 4.6.
template <int BITS, int LPGT, int MAXT, int HD>
__global__ void __launch_bounds__(MAXT)
k_attn_sites_fwd(SiteIns in, int64_t M, uint32_t S, const uint16_t* __restrict__ cosv, const uint16_t* __restrict__ sinv, int CPS) {
  constexpr int NSEG = Q<BITS>::NSEG, L = HD / 8;
  const SiteIn t = in.t[blockIdx.y];
  const ChanArgs& a = t.a;
  const int c = threadIdx.x;
  if (c >= CPS) return;                                 // (heads and scale groups never straddle the end of a segment)
  const int64_t SEG = (int64_t)CPS * 8, H = SEG * NSEG;
  const bool leader = (c & (LPGT - 1)) == 0, rotate = t.rows != nullptr, absmax = a.absmax != 0;
  const int seg_groups = CPS >> a.chunk_to_group_shift;
  uint32_t km[NSEG][4];
  {
    uint32_t plan[NSEG];
#pragma unroll
    for (int i = 0; i < NSEG; ++i) plan[i] = a.plan[i * CPS + c];
    ChunkOutliers<NSEG> co;
    co.init(plan);
#pragma unroll
    for (int i = 0; i < NSEG; ++i) co.keep_masks(i, km[i]);
  }
  const int d0 = 8 * (c & (L - 1));                     // the chunk's first channel within its head
  const uint32_t flip = d0 < HD / 2 ? 0x80000000u : 0u;
  // channel ch of row m, rotated
  auto one = [&](const uint16_t* xr, uint32_t s, int ch) __attribute__((always_inline)) {
    const uint16_t v = xr[ch];
    if (!rotate) return v;
    const int d = ch & (HD - 1);
    const float w = bf_to_f(xr[d < HD / 2 ? ch + HD / 2 : ch - HD / 2]) * bf_to_f(sinv[(int64_t)s * HD + d]);
    return f_to_bf(__builtin_fmaf(bf_to_f(v), bf_to_f(cosv[(int64_t)s * HD + d]), d < HD / 2 ? -w : w));
  };
  const bool gather = c < a.k;
  const int idx0 = gather ? a.idx[c] : 0;
  const int64_t stride = gridDim.x;
  uint4 raw[NSEG], nxt[NSEG], cs = make_uint4(0, 0, 0, 0), sn = cs, cs_n = cs, sn_n = cs;
  auto load = [&](int64_t row, uint4 (&r)[NSEG], uint4& cw, uint4& sw) __attribute__((always_inline)) {
    const uint16_t* xp = t.x + row * t.ldx + 8 * c;
#pragma unroll
    for (int i = 0; i < NSEG; ++i) r[i] = *reinterpret_cast<const uint4*>(xp + i * SEG);
    if (rotate) {
      const int64_t at = (int64_t)((uint32_t)row % S) * HD + d0;
      cw = *reinterpret_cast<const uint4*>(cosv + at);
      sw = *reinterpret_cast<const uint4*>(sinv + at);
    }
  };
  int64_t row = blockIdx.x;
  if (row < M) load(row, raw, cs, sn);
  for (; row < M; row += stride) {
    if (row + stride < M) load(row + stride, nxt, cs_n, sn_n);
    const uint16_t* xr = t.x + row * t.ldx;
    const uint32_t s = (uint32_t)row % S;
    uint16_t* vp = t.vals + row * a.k;
    if (gather) {
      vp[c] = one(xr, s, idx0);
      for (int u = c + CPS; u < a.k; u += CPS) vp[u] = one(xr, s, a.idx[u]);
    }
    if (rotate) {
      float cf[8], sf[8];
      unpack8(cs, cf);
      unpack8(make_uint4(sn.x ^ (flip | flip >> 16), sn.y ^ (flip | flip >> 16), sn.z ^ (flip | flip >> 16), sn.w ^ (flip | flip >> 16)), sf);
#pragma unroll
      for (int i = 0; i < NSEG; ++i) {
        float own[8], far[8];
        unpack8(raw[i], own);
        unpack8(make_uint4(other_half<HD>(raw[i].x), other_half<HD>(raw[i].y), other_half<HD>(raw[i].z), other_half<HD>(raw[i].w)), far);
#pragma unroll
        for (int j = 0; j < 8; ++j) own[j] = __builtin_fmaf(own[j], cf[j], far[j] * sf[j]);
        raw[i] = pack8(own);
        *reinterpret_cast<uint4*>(t.rows + row * H + i * SEG + 8 * c) = raw[i];       // (the attention reads them next)
      }
    }
    uint32_t lo = 0, hi = 0;
    uint16_t* scp = t.scales + row * a.groups_per_row + (c >> a.chunk_to_group_shift);
#pragma unroll
    for (int i = 0; i < NSEG; ++i) {
      float v[8];
      unpack8(make_uint4(raw[i].x & km[i][0], raw[i].y & km[i][1], raw[i].z & km[i][2], raw[i].w & km[i][3]), v);
      uint32_t cl, ch;
      const float sc = quant_seg<BITS, LPGT, SCALE_RUNTIME>(v, LPGT, cl, ch, absmax);
      if (leader) scp[i * seg_groups] = f_to_bf(sc);
      if (BITS == 8) { lo = cl; hi = ch; }
      else { lo |= cl << (i * BITS); hi |= ch << (i * BITS); }
    }
    { const u32x2_t w = {lo, hi}; __builtin_nontemporal_store(w, reinterpret_cast<u32x2_t*>(t.stored + row * SEG + 8 * c)); }
#pragma unroll
    for (int i = 0; i < NSEG; ++i) raw[i] = nxt[i];
    cs = cs_n; sn = sn_n;
  }
}

struct SiteOut {
  const uint8_t* stored;
  const uint16_t *vals, *scales;
  ChanArgs a;
  uint16_t* xhat;
};
struct SiteOuts { SiteOut t[4]; };
struct RowTerms {                                       // k_attn_delta's operands, out of the fourth tensor's codes
  const uint16_t* g;
  int64_t ldg;
  const float* lse;
  float *nlse, *ndelta;
  uint32_t S;
  int heads, rows;                                       // rows of a workgroup
  float inv_scale;
};

// k_decompress_chan_fast for q, k and v, and for the output, where there is one, the sums dO * O of its heads instead of its rows,
// with k_attn_delta's lanes and order.  Bound by memory: the restored output is neither written nor read.  In a layer of
// 4 x 1024 x 32 x 128, 4 bits: five launches of 62 us -> one of 45 (30 with the codes in the last-level cache, 21 for q, k and v
// alone); 157 x 16 x 128, 8 bits: 18.8 -> 4.8; without the output 1 x 2048 x 32 x 128: three launches of 22.6 us -> one of 19.9.
template <int BITS, int MAXT, int HD>
__global__ void __launch_bounds__(MAXT)
k_attn_sites_bwd(SiteOuts out, RowTerms d, int64_t M, int CPS) {
  constexpr int NSEG = Q<BITS>::NSEG, L = HD / 8;
  const SiteOut t = out.t[gridDim.y == 4 ? (blockIdx.y + 3) & 3 : blockIdx.y];
  const ChanArgs& a = t.a;
  const bool terms = blockIdx.y == 0 && gridDim.y == 4;         // (the longest first)
  const int c = threadIdx.x;
  if (c >= CPS) return;
  const int64_t SEG = (int64_t)CPS * 8, H = SEG * NSEG;
  const int seg_groups = CPS >> a.chunk_to_group_shift;
  uint32_t plan[NSEG];
#pragma unroll
  for (int i = 0; i < NSEG; ++i) plan[i] = a.plan[i * CPS + c];
  ChunkOutliers<NSEG> co;
  co.init(plan);
  struct Row { uint2 pk; uint32_t sc[NSEG], o0[NSEG], o1[NSEG]; uint4 g[NSEG]; };
  auto load = [&](int64_t row, Row& r) __attribute__((always_inline)) {
    r.pk = *reinterpret_cast<const uint2*>(t.stored + row * SEG + 8 * c);
    const uint16_t* scp = t.scales + row * a.groups_per_row + (c >> a.chunk_to_group_shift);
#pragma unroll
    for (int i = 0; i < NSEG; ++i) r.sc[i] = scp[i * seg_groups];
    co.request(t.vals + row * a.k, r.o0, r.o1);
    if (terms) {
#pragma unroll
      for (int i = 0; i < NSEG; ++i) r.g[i] = *reinterpret_cast<const uint4*>(d.g + row * d.ldg + i * SEG + 8 * c);
    }
  };
  // (the row terms of neighbouring rows lie side by side: one workgroup takes them, or the lines they fill travel between the L2s)
  const int64_t stride = terms ? 1 : gridDim.x, end = terms && (int64_t)(blockIdx.x + 1) * d.rows < M ? (int64_t)(blockIdx.x + 1) * d.rows : M;
  int64_t row = (int64_t)blockIdx.x * (terms ? d.rows : 1);
  Row now = {}, nxt = {};
  if (row < end) load(row, now);
  for (; row < end; row += stride) {
    if (row + stride < end) load(row + stride, nxt);
#pragma unroll
    for (int i = 0; i < NSEG; ++i) {
      const float sf = bf_to_f((uint16_t)now.sc[i]);
      uint4 r = co.splice(i, dequant8<BITS>(now.pk.x, now.pk.y, i, sf), now.o0[i], now.o1[i], sf);
      if (co.more_pairs) r = splice_more(r, co.more_pairs, a.plan[i * CPS + c], t.vals + row * a.k, true, sf);
      if (!terms) {
        store_stream(t.xhat + row * H + i * SEG + 8 * c, r);
        continue;
      }
      float g[8], o[8], v = 0.f;
      unpack8(now.g[i], g);
      unpack8(r, o);
#pragma unroll
      for (int j = 0; j < 8; ++j) v = __builtin_fmaf(g[j], o[j], v);
      v = group_reduce<L>(v, OpAdd());
      if ((c & (L - 1)) == 0) {
        const uint32_t b = (uint32_t)row / d.S, s = (uint32_t)row - b * d.S;
        const int64_t at = ((int64_t)b * d.heads + (i * CPS + c) / L) * d.S + s;
        d.ndelta[at] = -v;
        d.nlse[at] = -(d.lse[at] * d.inv_scale);
      }
    }
    now = nxt;
  }
}

// what the two entries cover: channel codes of 4 and 8 bits in groups of 64 or 128, one chunk a lane, whole heads of 64 or 128 channels
// in every segment
static int sites_args(const char* who, int64_t B, int64_t S, int64_t heads, int64_t hd, const hyc_desc* d, int n, RowGeom* g, ChanArgs* a) {
  if (B < 0 || S < 0 || heads <= 0 || heads > 65536 || hd <= 0) return fail(HYC_EINVAL, "%s: B=%lld S=%lld heads=%lld head_dim=%lld", who, (long long)B, (long long)S, (long long)heads, (long long)hd);
  if (hd != 64 && hd != 128) return fail(HYC_ENOTSUP, "%s: head_dim %lld (64 or 128)", who, (long long)hd);
  if (S > 0 && B > (((int64_t)1 << 31) - 1) / S) return fail(HYC_ENOTSUP, "%s: B*S must stay below 2^31", who);
  if (!d) return fail(HYC_EFAULT, "%s: null descriptor", who);
  const int64_t H = heads * hd;
  for (int i = 0; i < n; ++i) {
    if (d[i].mode != HYC_MODE_CHANNEL || d[i].bits != d[0].bits || d[i].group != d[0].group || (d[0].bits != 4 && d[0].bits != 8) ||
        (d[0].group != 64 && d[0].group != 128))
      return fail(HYC_ENOTSUP, "%s: channel codes of 4 or 8 bits in groups of 64 or 128, the same for all", who);
    int lpg, rc = row_geom(H, d[i].bits, g);
    if (!rc) rc = make_chan_args(&d[i], *g, &a[i], &lpg);
    if (rc) return rc;
  }
  if (g->iters != 1 || g->seg % hd != 0) return fail(HYC_ENOTSUP, "%s: rows of %lld channels", who, (long long)H);
  return HYC_OK;
}
// workgroups of one tensor: two rows each where there are rows for it (compress.hip's grids)
static unsigned sites_grid(int64_t M, int threads) {
  const int64_t most = threads >= 512 ? 768 : 2048, g = M < most ? M : most;
  return (unsigned)(M / 2 > g ? M / 2 : g);
}

}  // namespace hyc

using namespace hyc;

extern "C" {

int hyc_attn_sites_fwd(const void* const* x, const int64_t* ldx, const void* cosv, const void* sinv, int64_t B, int64_t S, int64_t heads,
                       int64_t head_dim, const hyc_desc* d, void* const* rows, void* const* stored, void* const* vals, void* const* scales,
                       void* stream) {
  RowGeom g;
  SiteIns in = {};
  ChanArgs a[3];
  int rc = sites_args("hyc_attn_sites_fwd", B, S, heads, head_dim, d, 3, &g, a);
  if (rc) return rc;
  const int64_t M = B * S;
  if (M == 0) return HYC_OK;
  if (!x || !ldx || !rows || !stored || !vals || !scales || !cosv || !sinv) return fail(HYC_EFAULT, "hyc_attn_sites_fwd: null buffer");
  if (!aligned16(cosv) || !aligned16(sinv)) return fail(HYC_EINVAL, "hyc_attn_sites_fwd: buffers must be 16-byte aligned");
  for (int i = 0; i < 3; ++i) {
    if (!x[i] || (i < 2 && !rows[i]) || !stored[i] || !scales[i] || (a[i].k > 0 && !vals[i])) return fail(HYC_EFAULT, "hyc_attn_sites_fwd: null buffer");
    if (!aligned16(x[i]) || !aligned16(rows[i]) || !aligned8(stored[i]) || ldx[i] < g.H || ldx[i] % 8 != 0)
      return fail(HYC_EINVAL, "hyc_attn_sites_fwd: rows must be 16-byte aligned, a multiple of 8 (at least heads*head_dim) apart");
    in.t[i] = {static_cast<const uint16_t*>(x[i]), ldx[i], i < 2 ? static_cast<uint16_t*>(rows[i]) : nullptr, static_cast<uint8_t*>(stored[i]),
               static_cast<uint16_t*>(vals[i]), static_cast<uint16_t*>(scales[i]), a[i]};
  }
  const dim3 grid(sites_grid(M, g.threads), 3), block((unsigned)g.threads);
  hipStream_t st = begin_launch(stream);
#define HYC_GO(B_, L_, T_, HD_)                                                                                                        \
  hipLaunchKernelGGL((k_attn_sites_fwd<B_, L_, T_, HD_>), grid, block, 0, st, in, M, (uint32_t)S, static_cast<const uint16_t*>(cosv), \
                     static_cast<const uint16_t*>(sinv), g.cps)
#define HYC_T(B_, L_, HD_) do { if (g.threads <= 256) HYC_GO(B_, L_, 256, HD_); else HYC_GO(B_, L_, 1024, HD_); } while (0)
#define HYC_HD(B_, L_) do { if (head_dim == 128) HYC_T(B_, L_, 128); else HYC_T(B_, L_, 64); } while (0)
  if (d->bits == 4) { if (d->group == 64) HYC_HD(4, 8); else HYC_HD(4, 16); }
  else if (d->group == 64) HYC_HD(8, 8);
  else HYC_HD(8, 16);
#undef HYC_HD
#undef HYC_T
#undef HYC_GO
  return check_launch("hyc_attn_sites_fwd");
}

int hyc_attn_sites_bwd(const void* const* stored, const void* const* vals, const void* const* scales, const hyc_desc* d, int32_t n, int64_t B,
                       int64_t S, int64_t heads, int64_t head_dim, void* const* xhat, const void* dout, int64_t ldg, const float* lse, float scale,
                       float* workspace, void* stream) {
  RowGeom g;
  SiteOuts out = {};
  RowTerms r = {};
  ChanArgs a[4];
  if (n != 3 && n != 4) return fail(HYC_EINVAL, "hyc_attn_sites_bwd: %d tensors (3 or 4)", n);
  int rc = sites_args("hyc_attn_sites_bwd", B, S, heads, head_dim, d, n, &g, a);
  if (rc) return rc;
  const int64_t M = B * S;
  if (M == 0) return HYC_OK;
  if (!stored || !vals || !scales || !xhat) return fail(HYC_EFAULT, "hyc_attn_sites_bwd: null buffer");
  for (int i = 0; i < n; ++i) {
    if (!stored[i] || !scales[i] || (a[i].k > 0 && !vals[i]) || (i < 3 && !xhat[i])) return fail(HYC_EFAULT, "hyc_attn_sites_bwd: null buffer");
    if (!aligned8(stored[i]) || (i < 3 && !aligned16(xhat[i]))) return fail(HYC_EINVAL, "hyc_attn_sites_bwd: xhat must be 16-byte and stored 8-byte aligned");
    out.t[i] = {static_cast<const uint8_t*>(stored[i]), static_cast<const uint16_t*>(vals[i]), static_cast<const uint16_t*>(scales[i]), a[i],
                i < 3 ? static_cast<uint16_t*>(xhat[i]) : nullptr};
  }
  if (n == 4) {
    if (!(scale > 0.f) || !(1.0f / scale < __builtin_inff())) return fail(HYC_EINVAL, "hyc_attn_sites_bwd: scale must be positive and finite, as its reciprocal");
    if (!dout || !lse || !workspace) return fail(HYC_EFAULT, "hyc_attn_sites_bwd: null buffer");
    if (!aligned16(dout) || ldg < g.H || ldg % 8 != 0) return fail(HYC_EINVAL, "hyc_attn_sites_bwd: dout must be 16-byte aligned, rows a multiple of 8 apart");
    r = {static_cast<const uint16_t*>(dout), ldg, lse, workspace, workspace + M * heads, (uint32_t)S, (int)heads,
         (int)(M >= 4096 ? 8 : M >= 512 ? M / 512 : 1), 1.0f / scale};
  }
  const int64_t across = sites_grid(M, g.threads), tall = n == 4 ? (M + r.rows - 1) / r.rows : 0;
  const dim3 grid((unsigned)(across > tall ? across : tall), (unsigned)n), block((unsigned)g.threads);
  hipStream_t st = begin_launch(stream);
#define HYC_GO(B_, T_, HD_) hipLaunchKernelGGL((k_attn_sites_bwd<B_, T_, HD_>), grid, block, 0, st, out, r, M, g.cps)
#define HYC_HD(B_, T_) do { if (head_dim == 128) HYC_GO(B_, T_, 128); else HYC_GO(B_, T_, 64); } while (0)
  if (d->bits == 4) { if (g.threads <= 256) HYC_HD(4, 256); else HYC_HD(4, 1024); }
  else if (g.threads <= 256) HYC_HD(8, 256);
  else HYC_HD(8, 1024);
#undef HYC_HD
#undef HYC_GO
  return check_launch("hyc_attn_sites_bwd");
}

}  // extern "C"
