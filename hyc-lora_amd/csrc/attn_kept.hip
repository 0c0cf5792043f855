// Causal attention that keeps its probabilities above a threshold for the backward: the reference's eager attention with its
// sparsified softmax (models/modeling_llama.py:423-462, operators/efficient_softmax.py:10-45), without an [S, S] matrix.
//
//   forward    out and lse as hyc_attn_fwd gives them; kept are the entries p = bf16(exp(scale q.k - lse)) > threshold, as CSR
//              rows with ascending columns (Ph)
//   backward   dp = dO V^T at the kept entries only, D = sum_j Ph dp, dS = Ph o (dp - D),
//              dV = Ph^T dO, dQ = scale dS K, dK = scale dS^T Q
//
// About 1 % of the square is kept, so what belongs to a query is walked entry by entry (rows of k and v gathered, 2 x 256 bytes
// an entry) and only what belongs to a key, a sum over all later queries, is a product of dense tiles, built in LDS from the
// entries of 32 queries.  Beside batched products over whole score matrices this leaves out the masked half and most of what
// multiplies zeros.  Attention alone, forward and backward with the compression of q, k and v, score matrices -> here, us: 1 x 2048
// x 32 heads x 128 with 1 / 3 / 6 % kept 907 -> 366, 898 -> 499, 934 -> 743; 4 x 512 x 32 x 64 667 -> 363, 1 x 64 x 8 x 128 675 ->
// 365 (both the host's time, any of these shares).
//
// Kernels at 1 x 2048 x 32 x 128, 1 % kept, us: forward 62, kept entries 52, their copy to the CSR arrays 11 (and 10 for offsets and
// rows that overflow), dQ 47, dK / dV 93.  The products of scores and of dK / dV are bound by LDS and the chain of a wave's steps:
// every wave reads whole tiles, 2 waves to a SIMD; dQ by its vector instructions (37 per entry and row of 16 lanes; with a wave per
// row, dQ's two sums in one walk, it took 93).  With tiles of 64 queries, single-buffered, dK / dV took 98.
#include "attn_tiles.hpp"
#include "softmax_slab.hpp"

namespace hyc {

constexpr int KEPT_MAX_S = 32768;        // a column number fits 16 bits with room

// The kept entries of 128 queries of one matrix per workgroup: scores again (the forward's are gone by the time a row's lse is
// known), one comparison per score, and for the few that pass the bf16 probability of the score rounded to bf16: scores are bf16
// tensors in the reference and wherever they are written out here, and which entries are kept depends on that rounding (1 to 2 %
// of them lie within it of the threshold).
// FILL false: counts, and the first `cap` entries of a row to slab + row cap (column low, bf16 bits high).
// FILL true: only rows of more than `cap` entries, straight to the CSR arrays (a workgroup without one leaves at once).
// A lane's scores go through 144 bytes of LDS of its own, from which the loop over its kept bits picks by number (a loop over
// registers cannot, and 32 predicated blocks are executed for nearly every one of them as soon as one lane of 64 needs it).
template <int HD, bool FILL>
__global__ void __launch_bounds__(256, 2)
k_attn_kept(AttnRows Q, AttnRows K, const float* __restrict__ lse, int S, int heads, int first, int BH, int blocks, float scale,
            float log2_limit, uint32_t least_bits, int32_t* __restrict__ counts, uint32_t* __restrict__ slab, int cap,
            const int32_t* __restrict__ row_ptr, int32_t* __restrict__ cols, uint16_t* __restrict__ vals) {
  constexpr int KS = HD / 16, LANE_F = 36;                              // floats of a lane's scores: 32 and 4 against bank conflicts
  __shared__ __align__(1024) uint16_t lds[2 * AT_WALK * HD];            // K tiles
  __shared__ __align__(16) float scores[256 * LANE_F];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hi = lane >> 5;
  int block, m;
  attn_block(blocks, BH, true, &block, &m);
  const int bh = first + m, b = bh / heads, h = bh - b * heads;
  const int q0 = block * AT_OWN, w0 = q0 + 32 * wave;
  const int my_q = w0 + (lane & 31);
  const bool live = my_q < S;
  const int64_t my_row = (int64_t)m * S + (live ? my_q : S - 1);
  bool need = live;
  int64_t out_at = my_row * cap;
  int room = cap;
  if (FILL) {
    need = live && counts[my_row] > cap;
    if (!__syncthreads_or(need)) return;
    out_at = row_ptr[my_row];
    room = row_ptr[my_row + 1] - (int)out_at;
  }
  auto rows_of = [&](const AttnRows& t) { return t.p + (int64_t)b * S * t.pitch + (int64_t)h * HD; };
  const u32x4_t rk = uniform_rsrc(rows_of(K), (uint32_t)(((int64_t)(S - 1) * K.pitch + HD) * 2));
  const uint32_t pk = (uint32_t)K.pitch * 2u, base = lds_offset(lds);
  constexpr uint32_t TB = AT_WALK * HD * 2;                             // bytes of a tile
  TileLane<HD> lane_at;
  lane_at.init(base);
  const int q_end = q0 + AT_OWN < S ? q0 + AT_OWN : S;
  const int tiles = (q_end + AT_WALK - 1) / AT_WALK;
  issue_tile<HD>(rk, pk, 0, S - 1, base);
  bf16x8_t qf[KS];
  load_own<HD>(rows_of(Q), (uint32_t)Q.pitch * 2u, w0, S - 1, qf);
  const float l2 = lse[(int64_t)bh * S + (live ? my_q : S - 1)] * LOG2E;
  // the comparison on the accumulators: the score at which p reaches the limit, between two bf16 values; the rounded score passes
  // where the unrounded one lies beyond the middle between those (an infinite lse makes a NaN of it: nothing passes)
  const float middle = __uint_as_float((__float_as_uint((log2_limit + l2) * LN2) & 0xFFFF0000u) | 0x8000u);
  const float limit = need ? middle / scale : INFINITY;
  float* mine_f = scores + threadIdx.x * LANE_F;
  int count = 0;
  for (int t = 0; t < tiles; ++t) {
    tile_barrier();
    if (t + 1 < tiles) issue_tile<HD>(rk, pk, (t + 1) * AT_WALK, S - 1, base + ((t + 1) & 1) * TB);
    const int k0 = t * AT_WALK;
    if (k0 > w0 + 31) continue;                                         // (the same for the whole wave) all of it above the diagonal
    const TileLane<HD> T = lane_at.in((t & 1) * TB);
    floatx16_t s[2] = {zero16(), zero16()};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) s[kb] = HYC_MFMA(frag_rows<HD>(T, 0, 32 * kb, ks), qf[ks], s[kb]);
    uint32_t mine[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      uint32_t bits = 0;                                                // bit = key of the 32: 8 (i / 4) + 4 hi + i % 4
#pragma unroll
      for (int i = 0; i < 16; ++i) bits |= s[kb][i] > limit ? 1u << (8 * (i >> 2) + (i & 3)) : 0u;
      const int d = my_q - k0 - 32 * kb;                                // keys 0 .. d are visible
      mine[kb] = (bits << (4 * hi)) & (d < 0 ? 0u : d >= 31 ? ~0u : (2u << d) - 1u);
    }
    if (!__ballot((mine[0] | mine[1]) != 0)) continue;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        *reinterpret_cast<floatx4_t*>(mine_f + 16 * kb + 4 * v) = floatx4_t{s[kb][4 * v], s[kb][4 * v + 1], s[kb][4 * v + 2], s[kb][4 * v + 3]};
    const uint32_t all0 = mine[0] | (uint32_t)__shfl_xor((int)mine[0], 32, 64), all1 = mine[1] | (uint32_t)__shfl_xor((int)mine[1], 32, 64);
    const int mid_count = count + __popc(all0);
    auto store = [&](float raw, int bit, int pos, int kb) __attribute__((always_inline)) {
      uint32_t p = f_to_bf(__builtin_amdgcn_exp2f(__builtin_fmaf(bfr(raw * scale), LOG2E, -l2)));
      p = p > least_bits ? p : least_bits;                              // (an fp32 rounding beside the threshold)
      const uint32_t col = (uint32_t)(k0 + 32 * kb + bit);
      if (pos < room) {
        if (FILL) {
          cols[out_at + pos] = (int32_t)col;
          vals[out_at + pos] = (uint16_t)p;
        } else {
          slab[out_at + pos] = col | (p << 16);
        }
      }
    };
    // (the two halves of the tile side by side: a trip is a chain of an LDS read, an exponential and a store)
    for (uint32_t w0 = mine[0], w1 = mine[1]; w0 | w1; w0 &= w0 - 1, w1 &= w1 - 1) {
      const int b0 = __builtin_ctz(w0 | 0x80000000u), b1 = __builtin_ctz(w1 | 0x80000000u);
      const float s0 = mine_f[4 * (b0 >> 3) + (b0 & 3)], s1 = mine_f[16 + 4 * (b1 >> 3) + (b1 & 3)];
      store(s0, b0, w0 ? count + __popc(all0 & ((1u << b0) - 1u)) : room, 0);
      store(s1, b1, w1 ? mid_count + __popc(all1 & ((1u << b1) - 1u)) : room, 1);
    }
    count = mid_count + __popc(all1);
  }
  if (!FILL && live && hi == 0) counts[my_row] = count;
}

// What belongs to a query: dp, D, dS and dQ.  HD / 8 lanes share a row (16 bytes each of every row they gather), so a wave takes 4 (8)
// neighbouring rows, entry by entry, and needs no sum across its rows.  dS = Ph (dp - D) needs D, the sum over the whole row, so
// the entries are walked twice, the rows of v the first and those of k the second time; in between dp waits in LDS (in the
// records behind the first PARK rounds).  The entries leave as records for k_attn_kept_dkdv: column | row % 64 << 16, Ph | bf16(dS) << 16.
template <int HD>
__global__ void __launch_bounds__(256)
k_attn_kept_dq(AttnRows K, AttnRows V, AttnRows G, const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ cols,
               const uint16_t* __restrict__ vals, const uint16_t* __restrict__ cosv, const uint16_t* __restrict__ sinv, AttnOut DQ,
               uint2* __restrict__ records, int S, int heads, int first, int BH, int row_blocks, float scale) {
  constexpr int L = HD / 8, E = 64 / L, UN = 4, PARK = 8;               // lanes and rows, steps in flight, rounds whose dp is in LDS
  __shared__ uint2 park_all[PARK][256];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & (L - 1), at0 = lane - c;
  // workgroups go to the eight XCDs in turn: with a multiple of 8 matrices an XCD walks its matrices one after the other, and the k
  // and v it gathers from stay in its L2
  int m, rb;
  if ((BH & 7) == 0) {
    const int x = blockIdx.x & 7, idx = blockIdx.x >> 3;
    m = (idx / row_blocks) * 8 + x;
    rb = idx % row_blocks;
  } else {
    m = blockIdx.x % BH;
    rb = blockIdx.x / BH;
  }
  const int i = (rb * 4 + wave) * E + lane / L;
  const bool live = i < S;
  const int bh = first + m, b = bh / heads, h = bh - b * heads;
  auto rows_of = [&](const AttnRows& t) { return t.p + (int64_t)b * S * t.pitch + (int64_t)h * HD; };
  const char* kb = reinterpret_cast<const char*>(rows_of(K));
  const char* vb = reinterpret_cast<const char*>(rows_of(V));
  const uint32_t pk = (uint32_t)K.pitch * 2u, pv = (uint32_t)V.pitch * 2u;
  float g[8];
  unpack8(*reinterpret_cast<const uint4*>(rows_of(G) + (int64_t)(live ? i : S - 1) * G.pitch + 8 * c), g);
  const int64_t row = (int64_t)m * S + (live ? i : S - 1);
  const int64_t e0 = row_ptr[row];
  const int n = live ? row_ptr[row + 1] - (int)e0 : 0;
  int most = n;
#pragma unroll
  for (int x = L; x < 64; x <<= 1) { const int o = __shfl_xor(most, x, 64); most = o > most ? o : most; }
  most = __builtin_amdgcn_readfirstlane(most);
  float D = 0.f;
  for (int at = 0, r = 0; at < most; at += L, ++r) {
    uint32_t w = 0;                                                     // the lane's entry: column | Ph
    if (at + c < n) {
      const int col = cols[e0 + at + c];
      w = (uint32_t)(col < S ? col : S - 1) | (uint32_t)vals[e0 + at + c] << 16;
    }
    float dp = 0.f;
    const int steps = most - at < L ? most - at : L;
    for (int it = 0; it < steps; it += UN) {
      uint4 vr[UN];
      float pe[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const uint32_t we = (uint32_t)__shfl((int)w, at0 + it + u, 64); // (it + u < L: UN divides L)
        vr[u] = make_uint4(0, 0, 0, 0);
        if (at + it + u < n) vr[u] = *reinterpret_cast<const uint4*>(vb + (uint64_t)((we & 0xFFFFu) * pv + 16u * c));
        pe[u] = bf_hi(we);
      }
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        float v[8];
        unpack8(vr[u], v);
        float d = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) d = __builtin_fmaf(g[j], v[j], d);
        d = group_reduce<L>(d, OpAdd());
        if (it + u == c) dp = d;
        D = __builtin_fmaf(pe[u], d, D);                                // (an entry past the row's: 0 times 0)
      }
    }
    const uint2 mine = make_uint2(w, __float_as_uint(dp));
    if (r < PARK) park_all[r][threadIdx.x] = mine;
    else if (at + c < n) records[e0 + at + c] = mine;
  }
  float t[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) t[j] = 0.f;
  for (int at = 0, r = 0; at < most; at += L, ++r) {
    uint2 mine = make_uint2(0u, 0u);
    if (r < PARK) mine = park_all[r][threadIdx.x];
    else if (at + c < n) mine = records[e0 + at + c];                   // (as this lane left them)
    const float p = bf_hi(mine.x), ds = p * (__uint_as_float(mine.y) - D);
    if (at + c < n)
      records[e0 + at + c] = make_uint2((mine.x & 0xFFFFu) | (uint32_t)(i & 63) << 16, (mine.x >> 16) | (uint32_t)f_to_bf(ds) << 16);
    const int steps = most - at < L ? most - at : L;
    for (int it = 0; it < steps; it += UN) {
      uint4 kr[UN];
      float de[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const uint32_t we = (uint32_t)__shfl((int)mine.x, at0 + it + u, 64);
        de[u] = __shfl(ds, at0 + it + u, 64);
        kr[u] = make_uint4(0, 0, 0, 0);
        if (at + it + u < n) kr[u] = *reinterpret_cast<const uint4*>(kb + (uint64_t)((we & 0xFFFFu) * pk + 16u * c));
        else de[u] = 0.f;
      }
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        float k[8];
        unpack8(kr[u], k);
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = __builtin_fmaf(de[u], k[j], t[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) t[j] *= scale;
  if (cosv) {                                                           // the gradient before the rotation, as store_own has it
    const int64_t at = (int64_t)(live ? i : S - 1) * HD + 8 * c;
    const bool low = c < L / 2;
    float cs[8], sn[8];
    unpack8(*reinterpret_cast<const uint4*>(cosv + at), cs);
    unpack8(*reinterpret_cast<const uint4*>(sinv + (low ? at + HD / 2 : at - HD / 2)), sn);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float o = xor_lane(t[j], L / 2);
      t[j] = __builtin_fmaf(t[j], cs[j], low ? o * sn[j] : -(o * sn[j]));
    }
  }
  if (live) *reinterpret_cast<uint4*>(DQ.p + ((int64_t)b * S + i) * DQ.pitch + (int64_t)h * HD + 8 * c) = pack8(t);
}

// What belongs to a key: dV = Ph^T dO and dK = scale dS^T Q.  A workgroup owns 128 keys (a wave 32, as columns of its accumulators) and
// walks the queries from the diagonal on in tiles of 32.  Their Ph and dS are built in LDS from the records, [key][query], queries
// of 16 in the order in which frag_cols delivers the other operand, so that a lane's operand is one 16-byte read (16-byte pieces
// swizzled over the keys: 16 lanes' reads use every bank once).  All tiles are double-buffered: while one is multiplied, the
// next Q and dO come in, the next Ph and dS are cleared (first half of the products) and filled (second half), and the records
// after that are requested.
constexpr int KD_WALK = 32;
template <int HD>
__global__ void __launch_bounds__(256, 2)
k_attn_kept_dkdv(AttnRows Q, AttnRows G, const int32_t* __restrict__ row_ptr, const uint2* __restrict__ records,
                 const uint16_t* __restrict__ cosv, const uint16_t* __restrict__ sinv, AttnOut DK, AttnOut DV, int S, int heads, int first,
                 int BH, int blocks, float scale) {
  constexpr int NB = HD / 32, NR = 3;                                   // records of a tile a thread holds
  constexpr int KIND = AT_OWN * KD_WALK;                                // elements of a Ph (dS) tile
  __shared__ __align__(1024) uint16_t lds[4 * KD_WALK * HD];            // [buffer][Q, dO]
  __shared__ __align__(1024) uint16_t sparse[4 * KIND];                 // [buffer][Ph, dS]
  __shared__ int bounds[KEPT_MAX_S / KD_WALK + 1];                      // where a tile's records start
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hi = lane >> 5;
  int block, m;
  attn_block(blocks, BH, false, &block, &m);
  const int bh = first + m, b = bh / heads, h = bh - b * heads;
  const int k0 = block * AT_OWN, w0 = k0 + 32 * wave;
  auto rows_of = [&](const AttnRows& t) { return t.p + (int64_t)b * S * t.pitch + (int64_t)h * HD; };
  auto bytes_of = [&](const AttnRows& t) { return (uint32_t)(((int64_t)(S - 1) * t.pitch + HD) * 2); };
  const u32x4_t rq = uniform_rsrc(rows_of(Q), bytes_of(Q)), rg = uniform_rsrc(rows_of(G), bytes_of(G));
  const uint32_t pq = (uint32_t)Q.pitch * 2u, pg = (uint32_t)G.pitch * 2u, base = lds_offset(lds);
  constexpr uint32_t TB = KD_WALK * HD * 2;
  TileLane<HD> lane_at;
  lane_at.init(base);
  const int t0 = k0 / KD_WALK, tiles = (S + KD_WALK - 1) / KD_WALK;
  const int32_t* rp = row_ptr + (int64_t)m * S;
  for (int t = t0 + (int)threadIdx.x; t <= tiles; t += 256) bounds[t] = rp[t * KD_WALK < S ? t * KD_WALK : S];
  __syncthreads();
  uint2 rec[NR];
  int lo = 0, end = 0;
  auto request = [&](int t) __attribute__((always_inline)) {
    lo = bounds[t < tiles ? t : tiles];
    end = bounds[t < tiles ? t + 1 : tiles];
#pragma unroll
    for (int u = 0; u < NR; ++u) {
      const int e = lo + (int)threadIdx.x + 256 * u;
      rec[u] = make_uint2(0xFFFFu, 0u);                                 // a column outside every block
      if (e < end) rec[u] = records[e];
    }
  };
  auto place = [&](const uint2& r, uint16_t* to) __attribute__((always_inline)) {
    const uint32_t key = (r.x & 0xFFFFu) - (uint32_t)k0;
    if (key < (uint32_t)AT_OWN) {
      const uint32_t q = r.x >> 16;                                     // queries of 16 as a lane reads them: {0-3, 8-11 | 4-7, 12-15}
      const uint32_t piece = ((q >> 3) & 2u) | ((q >> 2) & 1u);
      const uint32_t at = key * KD_WALK + ((piece ^ ((key >> 2) & 3u)) << 3) + ((q & 8u) >> 1) + (q & 3u);
      to[at] = (uint16_t)(r.y & 0xFFFFu);
      to[KIND + at] = (uint16_t)(r.y >> 16);
    }
  };
  auto clear = [&](uint16_t* to) __attribute__((always_inline)) {
#pragma unroll
    for (int z = 0; z < 2 * KIND / 2048; ++z) *reinterpret_cast<uint4*>(to + 8 * ((int)threadIdx.x + 256 * z)) = make_uint4(0, 0, 0, 0);
  };
  auto fill = [&](uint16_t* to) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NR; ++u) place(rec[u], to);
    for (int e = lo + (int)threadIdx.x + 256 * NR; e < end; e += 256) place(records[e], to);
  };
  auto fetch = [&](int t, int buf) __attribute__((always_inline)) {
    issue_tile<HD, KD_WALK>(rq, pq, t * KD_WALK, S - 1, base + buf * 2 * TB);
    issue_tile<HD, KD_WALK>(rg, pg, t * KD_WALK, S - 1, base + buf * 2 * TB + TB);
  };
  request(t0);
  fetch(t0, 0);
  clear(sparse);
  __syncthreads();
  fill(sparse);
  request(t0 + 1);
  floatx16_t dk[NB], dv[NB];
#pragma unroll
  for (int d = 0; d < NB; ++d) { dk[d] = zero16(); dv[d] = zero16(); }
  const uint32_t my_key = 32 * wave + (lane & 31);
  const uint16_t* own = sparse + my_key * KD_WALK;
  const uint32_t turn = (my_key >> 2) & 3u;
  for (int t = t0; t < tiles; ++t) {
    const int buf = (t - t0) & 1;
    tile_barrier();
    // (the records have arrived with the tile; said here, before the next tile is asked for, lest the compiler wait for that too)
#pragma unroll
    for (int u = 0; u < NR; ++u) asm volatile("" : "+v"(rec[u].x), "+v"(rec[u].y));
    uint16_t* next = sparse + (buf ^ 1) * 2 * KIND;
    const bool more = t + 1 < tiles;
    if (more) {
      fetch(t + 1, buf ^ 1);
      clear(next);
    }
    const bool mine = t * KD_WALK + KD_WALK - 1 >= w0;                  // (the same for the whole wave) not every query before the wave's keys
    const TileLane<HD> T = lane_at.in(buf * 2 * TB);                    // Q; dO is TB bytes behind
    auto products = [&](int ks) __attribute__((always_inline)) {
      const uint32_t at = buf * 2 * KIND + (((uint32_t)(2 * ks + hi) ^ turn) << 3);
      const bf16x8_t pf = *reinterpret_cast<const bf16x8_t*>(own + at);
      const bf16x8_t df = *reinterpret_cast<const bf16x8_t*>(own + KIND + at);
#pragma unroll
      for (int d = 0; d < NB; ++d) {
        dv[d] = HYC_MFMA(frag_cols<HD>(T, TB, 32 * d, 16 * ks), pf, dv[d]);
        dk[d] = HYC_MFMA(frag_cols<HD>(T, 0, 32 * d, 16 * ks), df, dk[d]);
      }
    };
    if (mine) products(0);
    __syncthreads();                                                    // `next` is clear
    if (more) {
      fill(next);
      request(t + 2);
    }
    if (mine) products(1);
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

static int kept_args(const char* who, int64_t B, int64_t S, int64_t heads, int64_t first, int64_t matrices) {
  if (S > KEPT_MAX_S) return fail(HYC_ENOTSUP, "%s: S=%lld (at most %d)", who, (long long)S, KEPT_MAX_S);
  if (first < 0 || matrices < 0 || first + matrices > B * heads)
    return fail(HYC_EINVAL, "%s: matrices %lld .. %lld of %lld", who, (long long)first, (long long)(first + matrices), (long long)(B * heads));
  if (matrices * S >= 0x7FFFFFFFll) return fail(HYC_ENOTSUP, "%s: %lld rows", who, (long long)(matrices * S));
  return HYC_OK;
}

// the comparison p > bf16 threshold on unrounded values: log2 of the largest fp32 value that still rounds to the threshold, and the
// bits of the next bf16 value above it
static int kept_limit(const char* who, float threshold, float* log2_limit, uint32_t* least_bits) {
  const float thr = round_to_bf16(threshold);
  if (!(thr > 1e-30f) || !(thr < 1.f)) return fail(HYC_ENOTSUP, "%s: threshold %g must be a normal number between 0 and 1", who, (double)threshold);
  uint32_t u;
  memcpy(&u, &thr, 4);
  *least_bits = (u >> 16) + 1;
  u += 0x8000u;                                             // halfway to the next: rounds to the even one of the two
  if ((u >> 16) & 1u) u -= 1u;
  float limit;
  memcpy(&limit, &u, 4);
  *log2_limit = (float)log2((double)limit);
  return HYC_OK;
}

template <bool FILL>
static void launch_kept(const void* q, int64_t ldq, const void* k, int64_t ldk, const float* lse, int64_t S, int64_t heads, int64_t head_dim,
                        float scale, float limit, uint32_t least, int64_t first, int64_t matrices, int32_t* counts, uint32_t* slab,
                        int64_t cap, const int32_t* row_ptr, int32_t* cols, void* vals, hipStream_t st) {
  const int blocks = (int)((S + AT_OWN - 1) / AT_OWN);
  const AttnRows Q{(const uint16_t*)q, ldq}, K{(const uint16_t*)k, ldk};
  const dim3 grid((unsigned)(blocks * matrices));
#define HYC_GO(HD_)                                                                                                                  \
  hipLaunchKernelGGL((k_attn_kept<HD_, FILL>), grid, dim3(256), 0, st, Q, K, lse, (int)S, (int)heads, (int)first, (int)matrices, blocks, \
                     scale, limit, least, counts, slab, (int)cap, row_ptr, cols, (uint16_t*)vals)
  if (head_dim == 128) HYC_GO(128);
  else HYC_GO(64);
#undef HYC_GO
}

}  // namespace hyc

using namespace hyc;

extern "C" {

int hyc_attn_kept(const void* q, int64_t ldq, const void* k, int64_t ldk, const float* lse, int64_t B, int64_t S, int64_t heads,
                  int64_t head_dim, float scale, float threshold, int64_t first, int64_t matrices, int32_t* counts, uint32_t* slab,
                  int64_t cap, void* stream) {
  const int64_t pitches[2] = {ldq, ldk};
  float limit;
  uint32_t least;
  int rc = attn_args("hyc_attn_kept", B, S, heads, head_dim, scale, pitches, 2);
  if (!rc) rc = kept_args("hyc_attn_kept", B, S, heads, first, matrices);
  if (!rc) rc = kept_limit("hyc_attn_kept", threshold, &limit, &least);
  if (rc) return rc;
  if (cap <= 0 || cap > S) return fail(HYC_EINVAL, "hyc_attn_kept: cap=%lld must be in 1..S=%lld", (long long)cap, (long long)S);
  if (matrices == 0 || S == 0) return HYC_OK;
  if (!q || !k || !lse || !counts || !slab) return fail(HYC_EFAULT, "hyc_attn_kept: null buffer");
  if (!aligned16(q) || !aligned16(k)) return fail(HYC_EINVAL, "hyc_attn_kept: q and k must be 16-byte aligned");
  launch_kept<false>(q, ldq, k, ldk, lse, S, heads, head_dim, scale, limit, least, first, matrices, counts, slab, cap, nullptr, nullptr,
                     nullptr, begin_launch(stream));
  return check_launch("hyc_attn_kept");
}

int hyc_attn_kept_fill(const void* q, int64_t ldq, const void* k, int64_t ldk, const float* lse, int64_t B, int64_t S, int64_t heads,
                       int64_t head_dim, float scale, float threshold, int64_t first, int64_t matrices, const int32_t* counts,
                       const uint32_t* slab, int64_t cap, const int32_t* row_ptr, int32_t* cols, void* vals, void* stream) {
  const int64_t pitches[2] = {ldq, ldk};
  float limit;
  uint32_t least;
  int rc = attn_args("hyc_attn_kept_fill", B, S, heads, head_dim, scale, pitches, 2);
  if (!rc) rc = kept_args("hyc_attn_kept_fill", B, S, heads, first, matrices);
  if (!rc) rc = kept_limit("hyc_attn_kept_fill", threshold, &limit, &least);
  if (rc) return rc;
  if (cap <= 0 || cap > S) return fail(HYC_EINVAL, "hyc_attn_kept_fill: cap=%lld must be in 1..S=%lld", (long long)cap, (long long)S);
  if (matrices == 0 || S == 0) return HYC_OK;
  if (!q || !k || !lse || !counts || !slab || !row_ptr || !cols || !vals) return fail(HYC_EFAULT, "hyc_attn_kept_fill: null buffer");
  if (!aligned16(q) || !aligned16(k)) return fail(HYC_EINVAL, "hyc_attn_kept_fill: q and k must be 16-byte aligned");
  hipStream_t st = begin_launch(stream);
  launch_slab_copy(matrices * S, counts, slab, cap, row_ptr, cols, vals, st);
  launch_kept<true>(q, ldq, k, ldk, lse, S, heads, head_dim, scale, limit, least, first, matrices, const_cast<int32_t*>(counts), nullptr, cap,
                    row_ptr, cols, vals, st);
  return check_launch("hyc_attn_kept_fill");
}

int hyc_attn_kept_bwd(const void* dout, int64_t ldg, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv,
                      const int32_t* row_ptr, const int32_t* cols, const void* vals, const void* cosv, const void* sinv, int64_t B,
                      int64_t S, int64_t heads, int64_t head_dim, float scale, int64_t first, int64_t matrices, void* dq, int64_t lddq,
                      void* dk, int64_t lddk, void* dv, int64_t lddv, void* records, void* stream) {
  const int64_t pitches[7] = {ldg, ldq, ldk, ldv, lddq, lddk, lddv};
  int rc = attn_args("hyc_attn_kept_bwd", B, S, heads, head_dim, scale, pitches, 7);
  if (!rc) rc = kept_args("hyc_attn_kept_bwd", B, S, heads, first, matrices);
  if (rc) return rc;
  if (matrices == 0 || S == 0) return HYC_OK;
  if (!dout || !q || !k || !v || !row_ptr || !cols || !vals || !records || !dq || !dk || !dv || ((cosv == nullptr) != (sinv == nullptr)))
    return fail(HYC_EFAULT, "hyc_attn_kept_bwd: null buffer");
  if (!aligned16(dout) || !aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(dq) || !aligned16(dk) || !aligned16(dv) ||
      !aligned8(records) || (cosv && (!aligned16(cosv) || !aligned16(sinv))))
    return fail(HYC_EINVAL, "hyc_attn_kept_bwd: buffers must be 16-byte aligned (records 8)");
  const int blocks = (int)((S + AT_OWN - 1) / AT_OWN), BH = (int)matrices, row_blocks = (int)((S + 4 * (512 / head_dim) - 1) / (4 * (512 / head_dim)));
  if ((int64_t)row_blocks * BH >= ((int64_t)1 << 24)) return fail(HYC_ENOTSUP, "hyc_attn_kept_bwd: %lld rows", (long long)(matrices * S));
  hipStream_t st = begin_launch(stream);
  const AttnRows Q{(const uint16_t*)q, ldq}, K{(const uint16_t*)k, ldk}, V{(const uint16_t*)v, ldv}, G{(const uint16_t*)dout, ldg};
  const AttnOut DQ{(uint16_t*)dq, lddq}, DK{(uint16_t*)dk, lddk}, DV{(uint16_t*)dv, lddv};
  uint2* rec = (uint2*)records;
#define HYC_GO(HD_)                                                                                                                \
  do {                                                                                                                             \
    hipLaunchKernelGGL((k_attn_kept_dq<HD_>), dim3((unsigned)(row_blocks * BH)), dim3(256), 0, st, K, V, G, row_ptr, cols,           \
                       (const uint16_t*)vals, (const uint16_t*)cosv, (const uint16_t*)sinv, DQ, rec, (int)S, (int)heads, (int)first,  \
                       BH, row_blocks, scale);                                                                                     \
    hipLaunchKernelGGL((k_attn_kept_dkdv<HD_>), dim3((unsigned)(blocks * BH)), dim3(256), 0, st, Q, G, row_ptr, rec,                 \
                       (const uint16_t*)cosv, (const uint16_t*)sinv, DK, DV, (int)S, (int)heads, (int)first, BH, blocks, scale);     \
  } while (0)
  if (head_dim == 128) HYC_GO(128);
  else HYC_GO(64);
#undef HYC_GO
  return check_launch("hyc_attn_kept_bwd");
}

}  // extern "C"
