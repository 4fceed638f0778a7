// Attention backward on gfx950 (replaces solution/k_attn.py:84-245): delta, dK/dV per query
// head, dQ; the shared layout and helpers are in attn_dev.h.
#include "attn_dev.h"

namespace {

// delta[h][t] = sum_d O[t][h][d] dO[t][h][d] (solution/k_attn.py:84-94): 16 lanes per (token, head)
__global__ __launch_bounds__(kAThreads) void attn_delta_kernel(const f16* __restrict__ o,
                                                               const f16* __restrict__ dout,
                                                               float* __restrict__ delta,
                                                               int64_t n_tokens, int nq) {
  const int64_t pair = (int64_t)blockIdx.x * (kAThreads / 16) + (threadIdx.x >> 4);
  if (pair >= n_tokens * nq) return;
  const int64_t t = pair / nq;
  const int hh = (int)(pair % nq), e = (threadIdx.x & 15) * 8;
  const int64_t off = t * nq * kHD + hh * kHD + e;
  const f16x8 ov = *reinterpret_cast<const f16x8*>(o + off);
  const f16x8 gv = *reinterpret_cast<const f16x8*>(dout + off);
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) s = __fadd_rn(s, __fmul_rn((float)ov[j], (float)gv[j]));
#pragma unroll
  for (int x = 1; x < 16; x <<= 1) s = __fadd_rn(s, __shfl_xor(s, x));
  if ((threadIdx.x & 15) == 0) delta[(int64_t)hh * n_tokens + t] = s;
}

// The tile ring of both backward kernels: a tile of two operands (kBN rows each) in one of four
// LDS stages, filled by LDS DMA.  Wave w's instruction i fills chunks (4 i + w) 64 + lane of an
// operand: row 16 i + 4 w + lane / 16, with a wave-uniform base per tile and a 32-bit offset per
// lane; rows past `rows` (the rows left in the sequence, less one) read that row (finite, masked
// to p = 0).
constexpr int kBwdStages = 4;
constexpr int kBwdLoads = kTileHalves / 8 / kAThreads;   // per operand per lane: 4
constexpr unsigned kStageBytes = kTileHalves * 2;

struct TileSource {
  uint64_t base;      // first row of tile 0
  unsigned rowb;      // bytes per row
  unsigned off0;      // this lane's offset for instruction 0
  unsigned chunk;     // this lane's (swizzled) chunk offset inside a row
};
__device__ __forceinline__ TileSource tile_source(const f16* base, int64_t row_halves, int wave,
                                                  int lane) {
  TileSource t;
  t.base = uniform64((uint64_t)base);
  t.rowb = (unsigned)(row_halves * (int64_t)sizeof(f16));
  const int r0 = 4 * wave + (lane >> 4);
  t.chunk = (unsigned)(((lane & 15) ^ swz16(r0)) << 4);
  t.off0 = (unsigned)r0 * t.rowb + t.chunk;
  return t;
}
__device__ __forceinline__ void tile_load(const TileSource& src, int64_t first_row, int rows,
                                          const f16* stage, int wave) {
  const uint64_t tb = src.base + (uint64_t)first_row * src.rowb;
  const unsigned last = (unsigned)(rows < kBN ? rows : kBN) * src.rowb + src.chunk;
#pragma unroll
  for (int i = 0; i < kBwdLoads; ++i) {
    const unsigned off = src.off0 + (unsigned)(16 * i) * src.rowb;
    dma16s(tb, off < last ? off : last,
           __builtin_amdgcn_readfirstlane(lds_addr(stage + (4 * i + wave) * 512)));
  }
}

// A barrier that orders the LDS DMA waited for before it, without a wait for the operand reads in
// flight (they are of stages that no load in flight touches).
__device__ __forceinline__ void tile_barrier() {
  wait_vmem<0>();
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Both backward kernels run one wave per SIMD (their accumulators and resident operands take most
// of its 512 registers), so what hides a wave's latencies is its own instruction order: tile t's
// step is 32 MFMAs of tile t + 1's two score products with one element of tile t's P and dS beside
// each, then the MFMAs that consume P and dS.  Every operand read stands four to six MFMAs before
// its use, also across the two phases and from step to step, and the one barrier of a step lies
// between the phases: after it, tile t - 1's stage takes tile t + 3, and tile t + 2 is readable.
// The order is held by scheduling barriers: left to itself the compiler waited for each operand
// read right before its MFMA.
// Measured on MI355X with the delta launch, 12 query / 2 KV heads (graph replays): one sequence of
// 8192 tokens 953 -> 741 us, of 2048 93.5 -> 70.8, 8 x 1024 186 -> 157, 4 x 512 41.3 -> 34.9.
constexpr int kAhead1 = 6, kAhead2 = 4;

// dQ (solution/k_attn.py:142-182): one workgroup per (block of kBM queries, query head), key
// tiles of kBN up to the diagonal
__device__ __forceinline__ void dq_block(const AttnArgs& a, int blk, int h,
                                         const f16* __restrict__ dout,
                                         const float* __restrict__ lse,
                                         const float* __restrict__ delta, float* __restrict__ dq,
                                         f16* Ks, f16* Vs) {
  int64_t s0;
  int seqlen, mstart;
  if (!block_of(a, blk, &s0, &seqlen, &mstart)) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, hl = lane >> 5, c = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(w);
  const int64_t ROW = (int64_t)(a.nq + 2 * a.nkv) * kHD, OROW = (int64_t)a.nq * kHD;
  const int kvh = h / (a.nq / a.nkv);
  const int m = mstart + 32 * w + c;
  const bool mval = m < seqlen && s0 + m < a.n_tokens;

  const int hi = mstart + kBM < seqlen ? mstart + kBM : seqlen;
  const int n_tiles = (hi + kBN - 1) / kBN;
  const TileSource ksrc = tile_source(a.qkv + s0 * ROW + (int64_t)(a.nq + kvh) * kHD, ROW, wave, lane);
  const TileSource vsrc = tile_source(a.qkv + s0 * ROW + (int64_t)(a.nq + a.nkv + kvh) * kHD, ROW, wave, lane);
  auto issue = [&](int t) {
    if (t >= n_tiles) return;
    const int st = t % kBwdStages;
    tile_load(ksrc, t * kBN, seqlen - 1 - t * kBN, Ks + st * kTileHalves, wave);
    tile_load(vsrc, t * kBN, seqlen - 1 - t * kBN, Vs + st * kTileHalves, wave);
  };
  issue(0);
  issue(1);
  issue(2);
  // this lane's query and dO rows and statistics, loaded at a clamped row and selected at once
  // (the compiler's wait for them stands here, not in the loop)
  f16x8 qf[kHD / 16], dof[kHD / 16];
  float lse_m, dl_m;
  {
    const int64_t rr = s0 + (mval ? m : mstart);
    const f16* qrow = a.qkv + rr * ROW + h * kHD + 8 * hl;
    const f16* drow = dout + rr * OROW + h * kHD + 8 * hl;
#pragma unroll
    for (int s = 0; s < kHD / 16; ++s) {
      qf[s] = *reinterpret_cast<const f16x8*>(qrow + 16 * s);
      dof[s] = *reinterpret_cast<const f16x8*>(drow + 16 * s);
    }
    lse_m = lse[(int64_t)h * a.n_tokens + rr];
    dl_m = delta[(int64_t)h * a.n_tokens + rr];
#pragma unroll
    for (int s = 0; s < kHD / 16; ++s) asm volatile("" : "+v"(qf[s]), "+v"(dof[s]));
    asm volatile("" : "+v"(lse_m), "+v"(dl_m));
#pragma unroll
    for (int s = 0; s < kHD / 16; ++s) {
      qf[s] = mval ? qf[s] : zero8();
      dof[s] = mval ? dof[s] : zero8();
    }
    lse_m = mval ? lse_m : 0.0f;
    dl_m = mval ? dl_m : 0.0f;
  }
  f32x16 dqacc[kHD / 32];
#pragma unroll
  for (int hb = 0; hb < kHD / 32; ++hb) dqacc[hb] = zero16();
  const unsigned krow = lds_addr(Ks) + row_base(lane), vrow = lds_addr(Vs) + row_base(lane);
  const unsigned kcol = lds_addr(Ks) + col_base(lane);
  // operand i of a tile's products: S^T = K Q^T and dP^T = V dO^T (keys kb * 32 + (row), queries
  // on the lanes): sub-step i / 4, dP^T for i / 2 odd, key half i % 2
  auto rd1 = [&](unsigned ka, unsigned va, int i) {
    return lds_read8((((i >> 1) & 1) ? va : ka) ^ (unsigned)(32 * (i >> 2)), (i & 1) * 32 * kHD * 2);
  };
  auto product = [&](f32x16 (&sacc)[2], f32x16 (&dpacc)[2], const f16x8& f, int i) {
    const int s = i >> 2, kb = i & 1;
    if ((i >> 1) & 1) dpacc[kb] = mfma(f, dof[s], s == 0 ? zero16() : dpacc[kb]);
    else sacc[kb] = mfma(f, qf[s], s == 0 ? zero16() : sacc[kb]);
  };
  f16x8 fr[kAhead1];
  // the wait for all three tiles costs no more than the query rows' own
  tile_barrier();
  f32x16 s_a[2], d_a[2], s_b[2], d_b[2];
  {
    const unsigned ka = fresh(krow), va = fresh(vrow);
#pragma unroll
    for (int i = 0; i < kAhead1; ++i) fr[i] = rd1(ka, va, i);
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      product(s_a, d_a, fr[i % kAhead1], i);
      if (i + kAhead1 < 32) fr[i % kAhead1] = rd1(ka, va, i + kAhead1);
      __builtin_amdgcn_sched_barrier(0);
    }
    const unsigned ka1 = fresh(krow + kStageBytes), va1 = fresh(vrow + kStageBytes);
#pragma unroll
    for (int i = 0; i < kAhead1; ++i) fr[i] = rd1(ka1, va1, i);
  }
  auto step = [&](int t, f32x16 (&sc)[2], f32x16 (&dc)[2], f32x16 (&sn)[2], f32x16 (&dn)[2],
                  auto more_c) {
    constexpr bool MORE = decltype(more_c)::value;   // tile t + 1 exists
    const int n0 = t * kBN;
    // keys past a query or the sequence are masked only on the tiles that reach this wave's first
    // query (a wave-uniform test): key n = n0 + off + 4 (l / 32) is kept iff
    // off <= min(m, seqlen - 1) - n0 - 4 (l / 32); the others' probabilities come out as 0.
    // Rows past the sequence have zero q, dO and delta, so their dS is zero whatever P is.
    if (n0 + kBN - 1 > mstart + 32 * wave || n0 + kBN > seqlen) {
      const int lim = (m < seqlen - 1 ? m : seqlen - 1) - n0 - 4 * hl;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          sc[kb][v] = kb * 32 + 8 * (v >> 2) + (v & 3) <= lim ? sc[kb][v] : -1.0e30f;
    }
    const unsigned nst = (unsigned)((t + 1) % kBwdStages) * kStageBytes;
    const unsigned ka = fresh(krow + nst), va = fresh(vrow + nst);
    const unsigned kc = fresh(kcol + (unsigned)(t % kBwdStages) * kStageBytes);
    auto rd2 = [&](int i) { return lds_col8(kc, i & 3, 16 * (i >> 2) * kHD * 2); };
    Frag8 dsf[kBN / 16];
    f16x8 gr[kAhead2];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      if constexpr (MORE) {
        product(sn, dn, fr[i % kAhead1], i);
        if (i + kAhead1 < 32) fr[i % kAhead1] = rd1(ka, va, i + kAhead1);
      }
      const int kb = i >> 4, v = i & 15;
      const float p = ex2(__builtin_fmaf(sc[kb][v], a.qk_scale, -lse_m));
      dc[kb][v] = __fmul_rn(p, __fsub_rn(dc[kb][v], dl_m));
      if (i & 1) dsf[i >> 3].h[(i >> 1) & 3] = pinned(dc[kb][v - 1], dc[kb][v]);
      if (i >= 32 - kAhead2) gr[i - (32 - kAhead2)] = rd2(i - (32 - kAhead2));
      if constexpr (MORE) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (MORE) {
      tile_barrier();
      issue(t + 3);
    }
    const unsigned nst2 = (unsigned)((t + 2) % kBwdStages) * kStageBytes;
    const unsigned ka2 = fresh(krow + nst2), va2 = fresh(vrow + nst2);
    // dQ^T += K^T dS^T
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      dqacc[i & 3] = mfma(gr[i % kAhead2], dsf[i >> 2].get(), dqacc[i & 3]);
      if (i + kAhead2 < 16) gr[i % kAhead2] = rd2(i + kAhead2);
      // (past the last tile: a stale stage, never used)
      if (MORE && i >= 16 - kAhead1) fr[i - (16 - kAhead1)] = rd1(ka2, va2, i - (16 - kAhead1));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using More = std::integral_constant<bool, true>;
  using Last = std::integral_constant<bool, false>;
  int t = 0;
  for (; t + 2 < n_tiles; t += 2) {
    step(t, s_a, d_a, s_b, d_b, More{});
    step(t + 1, s_b, d_b, s_a, d_a, More{});
  }
  if (t + 1 < n_tiles) {
    step(t, s_a, d_a, s_b, d_b, More{});
    ++t;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      s_a[kb] = s_b[kb];
      d_a[kb] = d_b[kb];
    }
  }
  step(t, s_a, d_a, s_b, d_b, Last{});
  __syncthreads();
  // the wave's 32 x 128 block of dQ staged in the (now free) tile ring, waves 0-1 in the K stages
  // and 2-3 in the V stages, then written back 16 bytes per lane, two whole 512-byte rows per
  // store instruction (stored from the registers, each instruction would cover 32 bytes of each
  // of 32 rows' cache lines); rows past the sequence are not stored
  constexpr int kQStride = kHD + 4;   // floats per staged row
  static_assert(2 * 32 * kQStride * 4 <= kFwdStages * kTileHalves * 2, "dQ staging in the ring");
  float* qstage = reinterpret_cast<float*>(w < 2 ? Ks : Vs) + (w & 1) * 32 * kQStride;
#pragma unroll
  for (int hb = 0; hb < kHD / 32; ++hb)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = __fmul_rn(dqacc[hb][4 * g + e], a.sm_scale);
      *reinterpret_cast<f32x4*>(qstage + c * kQStride + hb * 32 + 8 * g + 4 * hl) = o;
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = 2 * i + hl, row = mstart + 32 * w + r;
    const f32x4 v = *reinterpret_cast<const f32x4*>(qstage + r * kQStride + 4 * c);
    if (row < seqlen && s0 + row < a.n_tokens)
      *reinterpret_cast<f32x4*>(dq + (s0 + row) * OROW + h * kHD + 4 * c) = v;
  }
}

// dK, dV per query head (solution/k_attn.py:97-139): one workgroup per (block of kBM keys, query
// head), query tiles of kBN from the block's first key to the end of the sequence; fp32 partials
// [N, NQ HD] that the QKV epilogue backward sums over each group of NQ / NKV heads.  The Q and dO
// tiles and the tiles' lse and delta rows (by dword DMA, one lane per query, waves 0 and 1) come
// through the four-stage ring.
__device__ __forceinline__ void dkdv_block(const AttnArgs& a, int blk, int h,
                                           const f16* __restrict__ dout,
                                           const float* __restrict__ lse,
                                           const float* __restrict__ delta,
                                           float* __restrict__ dkp, float* __restrict__ dvp,
                                           f16* Qs, f16* Ds, float (*lse_s)[kBN],
                                           float (*dl_s)[kBN]) {
  int64_t s0;
  int seqlen, nstart;
  if (!block_of(a, blk, &s0, &seqlen, &nstart)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, hl = lane >> 5, c = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(w);
  const int64_t ROW = (int64_t)(a.nq + 2 * a.nkv) * kHD, OROW = (int64_t)a.nq * kHD;
  const int kvh = h / (a.nq / a.nkv);
  const int n = nstart + 32 * w + c;   // this lane's key
  const bool nval = n < seqlen && s0 + n < a.n_tokens;

  const int n_tiles = (seqlen - nstart + kBN - 1) / kBN;   // at least 1 (block_of)
  if ((int)threadIdx.x < kBN) lse_s[kBwdStages][threadIdx.x] = 0.0f;
  const TileSource qsrc = tile_source(a.qkv + (s0 + nstart) * ROW + (int64_t)h * kHD, ROW, wave, lane);
  const TileSource dsrc = tile_source(dout + (s0 + nstart) * OROW + (int64_t)h * kHD, OROW, wave, lane);
  // query tile t (queries nstart + 64 t ...); wave 0 also fetches the tile's lse, wave 1 its delta
  auto issue = [&](int t) {
    if (t >= n_tiles) return;
    const int st = t % kBwdStages, m0 = nstart + t * kBN;
    tile_load(qsrc, t * kBN, seqlen - 1 - m0, Qs + st * kTileHalves, wave);
    tile_load(dsrc, t * kBN, seqlen - 1 - m0, Ds + st * kTileHalves, wave);
    if (wave < 2) {
      const int qq = m0 + lane < seqlen ? m0 + lane : seqlen - 1;
      const float* src = (wave == 0 ? lse : delta) + (int64_t)h * a.n_tokens + s0 + qq;
      dma4(src, __builtin_amdgcn_readfirstlane(lds_addr(wave == 0 ? lse_s[st] : dl_s[st])));
    }
  };
  issue(0);
  issue(1);
  issue(2);

  // this lane's key and value rows as B operands, loaded at a clamped row and selected at once
  // (the compiler's wait for them stands here, not in the loop)
  f16x8 kf[kHD / 16], vf[kHD / 16];
  {
    const int64_t rr = s0 + (nval ? n : nstart);
    const f16* krow = a.qkv + rr * ROW + (int64_t)(a.nq + kvh) * kHD + 8 * hl;
    const f16* vrow = a.qkv + rr * ROW + (int64_t)(a.nq + a.nkv + kvh) * kHD + 8 * hl;
#pragma unroll
    for (int s = 0; s < kHD / 16; ++s) {
      kf[s] = *reinterpret_cast<const f16x8*>(krow + 16 * s);
      vf[s] = *reinterpret_cast<const f16x8*>(vrow + 16 * s);
    }
#pragma unroll
    for (int s = 0; s < kHD / 16; ++s) asm volatile("" : "+v"(kf[s]), "+v"(vf[s]));
#pragma unroll
    for (int s = 0; s < kHD / 16; ++s) {
      kf[s] = nval ? kf[s] : zero8();
      vf[s] = nval ? vf[s] : zero8();
    }
  }
  f32x16 dkacc[kHD / 32], dvacc[kHD / 32];
#pragma unroll
  for (int hb = 0; hb < kHD / 32; ++hb) dkacc[hb] = dvacc[hb] = zero16();
  const unsigned qrow = lds_addr(Qs) + row_base(lane), drow = lds_addr(Ds) + row_base(lane);
  const unsigned qcol = lds_addr(Qs) + col_base(lane), dcol = lds_addr(Ds) + col_base(lane);
  // operand i of a tile's products S = Q K^T and dP = dO V^T (queries qb * 32 + (row of the
  // result), keys on the lanes): sub-step i / 4, dP for i / 2 odd, query half i % 2
  auto rd1 = [&](unsigned qa, unsigned da, int i) {
    return lds_read8((((i >> 1) & 1) ? da : qa) ^ (unsigned)(32 * (i >> 2)), (i & 1) * 32 * kHD * 2);
  };
  auto product = [&](f32x16 (&sacc)[2], f32x16 (&dpacc)[2], const f16x8& f, int i) {
    const int s = i >> 2, qb = i & 1;
    if ((i >> 1) & 1) dpacc[qb] = mfma(f, vf[s], s == 0 ? zero16() : dpacc[qb]);
    else sacc[qb] = mfma(f, kf[s], s == 0 ? zero16() : sacc[qb]);
  };
  // the statistics of rows 8 g + 4 (l / 32) + 0..3 of the tile in stage st (g = 0..7)
  auto stat = [&](const float (*tab)[kBN], int st, int g) {
    return *reinterpret_cast<const f32x4*>(&tab[st][8 * g + 4 * hl]);
  };
  f16x8 fr[kAhead1];
  f32x4 ls[2], dl[2];
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the row of zeros is written
  tile_barrier();
  f32x16 s_a[2], d_a[2], s_b[2], d_b[2];
  {
    const unsigned qa = fresh(qrow), da = fresh(drow);
#pragma unroll
    for (int i = 0; i < kAhead1; ++i) fr[i] = rd1(qa, da, i);
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      product(s_a, d_a, fr[i % kAhead1], i);
      if (i + kAhead1 < 32) fr[i % kAhead1] = rd1(qa, da, i + kAhead1);
      __builtin_amdgcn_sched_barrier(0);
    }
    const unsigned qa1 = fresh(qrow + kStageBytes), da1 = fresh(drow + kStageBytes);
#pragma unroll
    for (int i = 0; i < kAhead1; ++i) fr[i] = rd1(qa1, da1, i);
    ls[0] = stat(lse_s, 0, 0);
    dl[0] = stat(dl_s, 0, 0);
  }
  auto step = [&](int t, f32x16 (&sc)[2], f32x16 (&dc)[2], f32x16 (&sn)[2], f32x16 (&dn)[2],
                  auto more_c) {
    constexpr bool MORE = decltype(more_c)::value;   // tile t + 1 exists
    const int st = t % kBwdStages, m0 = nstart + t * kBN;
    // Keys past the sequence only reach rows of dK and dV that are not stored; queries before a
    // key or past the sequence are masked only on the tiles that hold such a query for this wave
    // (a wave-uniform test): query q = m0 + off + 4 (l / 32) is kept iff lo <= off < hi.  There the
    // exponent is formed before the selection and the loop below is given scale 1 and a row of
    // zeros for lse, so that the others' probabilities are 0 whatever their lse is: a NaN query
    // reaches dV of no later key (masking the score alone would give e^NaN).
    float scale = a.qk_scale;
    int lrow = st;
    if (m0 < nstart + 32 * wave + 31 || m0 + kBN > seqlen) {
      const int lo = n - m0 - 4 * hl, hi = seqlen - m0 - 4 * hl;
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        const f32x4 l = g == 0 ? ls[0] : stat(lse_s, st, g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int off = 8 * g + e;
          const float x = __builtin_fmaf(sc[g >> 2][4 * (g & 3) + e], a.qk_scale, -l[e]);
          sc[g >> 2][4 * (g & 3) + e] = ((off >= lo) & (off < hi)) ? x : -1.0e30f;
        }
      }
      scale = 1.0f;
      lrow = kBwdStages;
      ls[0] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const unsigned nst = (unsigned)((t + 1) % kBwdStages) * kStageBytes;
    const unsigned qa = fresh(qrow + nst), da = fresh(drow + nst);
    const unsigned qc = fresh(qcol + (unsigned)st * kStageBytes), dc_ = fresh(dcol + (unsigned)st * kStageBytes);
    auto rd2 = [&](int i) { return lds_col8((i & 1) ? qc : dc_, (i >> 1) & 3, 16 * (i >> 3) * kHD * 2); };
    Frag8 pf[kBN / 16], dsf[kBN / 16];
    f16x8 gr[kAhead2];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      if constexpr (MORE) {
        product(sn, dn, fr[i % kAhead1], i);
        if (i + kAhead1 < 32) fr[i % kAhead1] = rd1(qa, da, i + kAhead1);
      }
      const int qb = i >> 4, v = i & 15, g = i >> 2;
      if ((i & 3) == 0 && g + 1 < 8) {
        ls[(g + 1) & 1] = stat(lse_s, lrow, g + 1);
        dl[(g + 1) & 1] = stat(dl_s, st, g + 1);
      }
      sc[qb][v] = ex2(__builtin_fmaf(sc[qb][v], scale, -ls[g & 1][i & 3]));
      dc[qb][v] = __fmul_rn(sc[qb][v], __fsub_rn(dc[qb][v], dl[g & 1][i & 3]));
      if (i & 1) {
        pf[i >> 3].h[(i >> 1) & 3] = pinned(sc[qb][v - 1], sc[qb][v]);
        dsf[i >> 3].h[(i >> 1) & 3] = pinned(dc[qb][v - 1], dc[qb][v]);
      }
      if (i >= 32 - kAhead2) gr[i - (32 - kAhead2)] = rd2(i - (32 - kAhead2));
      if constexpr (MORE) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (MORE) {
      tile_barrier();
      issue(t + 3);
    }
    const unsigned nst2 = (unsigned)((t + 2) % kBwdStages) * kStageBytes;
    const unsigned qa2 = fresh(qrow + nst2), da2 = fresh(drow + nst2);
    // dV += P^T dO, dK += dS^T Q over the tile's 64 queries, 16 per step
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const int hb = (i >> 1) & 3;
      if (i & 1) dkacc[hb] = mfma(dsf[i >> 3].get(), gr[i % kAhead2], dkacc[hb]);
      else dvacc[hb] = mfma(pf[i >> 3].get(), gr[i % kAhead2], dvacc[hb]);
      if (i + kAhead2 < 32) gr[i % kAhead2] = rd2(i + kAhead2);
      if constexpr (MORE) {
        // (past the last tile: a stale stage, never used)
        if (i >= 32 - kAhead1) fr[i - (32 - kAhead1)] = rd1(qa2, da2, i - (32 - kAhead1));
        if (i == 28) ls[0] = stat(lse_s, (t + 1) % kBwdStages, 0);
        if (i == 29) dl[0] = stat(dl_s, (t + 1) % kBwdStages, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using More = std::integral_constant<bool, true>;
  using Last = std::integral_constant<bool, false>;
  int t = 0;
  for (; t + 2 < n_tiles; t += 2) {
    step(t, s_a, d_a, s_b, d_b, More{});
    step(t + 1, s_b, d_b, s_a, d_a, More{});
  }
  if (t + 1 < n_tiles) {
    step(t, s_a, d_a, s_b, d_b, More{});
    ++t;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      s_a[qb] = s_b[qb];
      d_a[qb] = d_b[qb];
    }
  }
  step(t, s_a, d_a, s_b, d_b, Last{});
  // result register v of block hb: key 32 w + 8 (v / 4) + 4 (l / 32) + v % 4, column hb * 32 + c
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int key = nstart + 32 * w + 8 * (v >> 2) + 4 * hl + (v & 3);
    if (key >= seqlen || s0 + key >= a.n_tokens) continue;
    const int64_t off = (s0 + key) * OROW + h * kHD + c;
#pragma unroll
    for (int hb = 0; hb < kHD / 32; ++hb) {
      dkp[off + hb * 32] = __fmul_rn(dkacc[hb][v], a.sm_scale);
      dvp[off + hb * 32] = dvacc[hb][v];
    }
  }
}

// dK/dV and dQ in one launch.  Workgroups [0, n_blocks * nq) run the dK/dV blocks in block-table
// order, the rest the dQ blocks in reverse block-table order, each with every head of a block
// before the next block.  The hardware deals workgroups to the 8 XCDs round-robin and each XCD
// starts its own in index order, so with a table whose blocks are ordered by the rows from their
// start to their sequence's end, longest first (the dK/dV walk; reversed, the dQ walk for sequences
// of equal length), every XCD gets a balanced share, started longest first: the dQ blocks begin
// on the CUs the dK/dV blocks leave idle and then on those that short blocks free.  Any table
// order gives the same results.  Both read delta, which the launch before computes.
__global__ __launch_bounds__(kAThreads) void attn_bwd_kernel(AttnArgs a, const f16* __restrict__ dout,
                                                             const float* __restrict__ lse,
                                                             const float* __restrict__ delta,
                                                             float* __restrict__ dq,
                                                             float* __restrict__ dkp,
                                                             float* __restrict__ dvp, int n_blocks) {
  static_assert(kBwdStages == kFwdStages, "dK/dV and dQ share the tile ring");
  __shared__ __attribute__((aligned(1024))) f16 T0[kBwdStages * kTileHalves];
  __shared__ __attribute__((aligned(1024))) f16 T1[kBwdStages * kTileHalves];
  __shared__ __attribute__((aligned(16))) float lse_s[kBwdStages + 1][kBN], dl_s[kBwdStages][kBN];
  const int per = n_blocks * a.nq;
  const int g = blockIdx.x;
  if (g < per)
    dkdv_block(a, g / a.nq, g % a.nq, dout, lse, delta, dkp, dvp, T0, T1, lse_s, dl_s);
  else
    dq_block(a, n_blocks - 1 - (g - per) / a.nq, (g - per) % a.nq, dout, lse, delta, dq, T0, T1);
}

}  // namespace

extern "C" int dk_attn_bwd(const void* qkv, const void* out, const float* lse, const void* dout,
                           const int32_t* cu_seqlens, int32_t n_seq, const int32_t* block_table,
                           int32_t n_blocks, int64_t n_tokens, int32_t nq, int32_t nkv, int32_t hd,
                           float* delta, float* dq, float* dkp, float* dvp, hipStream_t stream) {
  AttnArgs a;
  if (int e = attn_args(a, qkv, cu_seqlens, n_seq, block_table, n_blocks, n_tokens, nq, nkv, hd))
    return e;
  if (n_blocks == 0 || n_tokens == 0) return 0;
  if (!out || !lse || !dout || !delta || !dq || !dkp || !dvp) return DK_ERR_INVALID;
  if (2 * (int64_t)n_blocks * nq > INT32_MAX) return DK_ERR_INVALID;   // one workgroup index
  if (!dk_aligned(out, 16) || !dk_aligned(dout, 16) || !dk_aligned(lse, 4) ||
      !dk_aligned(delta, 4) || !dk_aligned(dq, 16) || !dk_aligned(dkp, 4) || !dk_aligned(dvp, 4))
    return DK_ERR_ALIGN;
  const int64_t pairs = n_tokens * nq;
  hipLaunchKernelGGL(attn_delta_kernel, dim3((unsigned)((pairs + 15) / 16)), dim3(kAThreads), 0,
                     stream, (const f16*)out, (const f16*)dout, delta, n_tokens, nq);
  DK_CHECK_LAUNCH();
  hipLaunchKernelGGL(attn_bwd_kernel, dim3((unsigned)(2 * n_blocks * nq)), dim3(kAThreads), 0,
                     stream, a, (const f16*)dout, lse, delta, dq, dkp, dvp, n_blocks);
  DK_CHECK_LAUNCH();
  return 0;
}
