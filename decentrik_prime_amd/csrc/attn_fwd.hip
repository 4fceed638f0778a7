// Attention forward on gfx950 (replaces solution/k_attn.py:40-83): causal GQA over the packed
// sequences with an online softmax in the exp2 domain.  Built with the MFMA accumulators in
// VGPRs (the build passes -amdgpu-mfma-vgpr-form for this file): in AGPRs the compiler copied
// the output accumulator out and back on every key tile.
#include "attn_dev.h"

namespace {

// forward (solution/k_attn.py:40-83): one workgroup per (block of kBM queries, query head), 8
// waves: wave w takes queries 32 (w % 4) .. + 31 of the block and the key tiles t with
// t % 2 == w / 4, so two waves share each SIMD and each walks half of the block's tiles.  The two
// halves' softmax states (running maximum, sum, O) are merged through LDS at the end.
//
// Bound: per tile of 64 keys a wave has 32 MFMAs (1024 clocks of its SIMD's matrix core), 48 LDS
// operand reads and about 130 VALU instructions (32 of them quarter-rate exponentials).  One
// after the other these ran at a quarter of the matrix rate, with both waves of a SIMD in the same
// phase after every barrier.  So the scores of the wave's next tile are computed beside the
// exponentials of the current one (S(t + 2) needs nothing of tile t), and the K ring runs a
// pair of tiles ahead of the V ring.  Measured on MI355X, 12 query / 2 KV heads (graph replays): one
// sequence of 8192 tokens 417 -> 257 us (802 TFLOP/s), of 2048 40.9 -> 36.8, 8 x 1024 73.6 -> 62.0,
// 4 x 512 16.6 as before.
constexpr int kFThreads = 512;
constexpr int kFLoads = kTileHalves / 8 / kFThreads;   // DMA instructions per operand per lane: 2

// max over the two lanes l, l ^ 32 (the two key halves of one query)
__device__ __forceinline__ float half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__global__ __launch_bounds__(kFThreads) void attn_fwd_kernel(AttnArgs a, f16* __restrict__ out,
                                                             float* __restrict__ lse, int n_blocks) {
  // every head of a block before the next block, the table from its end: within a sequence the
  // longest walks start first, so that no long block is left to run alone at the end.  The grid is
  // n_blocks x nq (one dimension of n_blocks nq workgroups would end at 2^32 work items, 699,050
  // one-token sequences of 12 heads), its workgroups taken in launch order
  const int g = (int)(blockIdx.y * (unsigned)n_blocks + blockIdx.x);
  const int h = g % a.nq;
  int64_t s0;
  int seqlen, mstart;
  if (!block_of(a, n_blocks - 1 - g / a.nq, &s0, &seqlen, &mstart)) return;
  const int lane = threadIdx.x & 63, hl = lane >> 5, c = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int qw = wave & 3, kg = wave >> 2;   // query group, key-tile parity
  const int64_t ROW = (int64_t)(a.nq + 2 * a.nkv) * kHD;
  const int kvh = h / (a.nq / a.nkv);
  const int m = mstart + 32 * qw + c;
  const bool mval = m < seqlen && s0 + m < a.n_tokens;
  __shared__ __attribute__((aligned(1024))) f16 Ks[kFwdStages * kTileHalves];
  __shared__ __attribute__((aligned(1024))) f16 Vs[kFwdStages * kTileHalves];

  f32x16 oacc[kHD / 32];
#pragma unroll
  for (int hb = 0; hb < kHD / 32; ++hb) oacc[hb] = zero16();
  float m_i = -1.0e30f, l_i = 0.0f;   // l_i: this lane's half of the keys (joined at the end)
  const int hi = mstart + kBM < seqlen ? mstart + kBM : seqlen;
  const int n_tiles = (hi + kBN - 1) / kBN;
  const int n_pairs = (n_tiles + 1) / 2;
  const uint64_t kbase = uniform64((uint64_t)(a.qkv + s0 * ROW + (int64_t)(a.nq + kvh) * kHD));
  const uint64_t vbase = kbase + (uint64_t)a.nkv * kHD * sizeof(f16);
  // tile pair u (tiles 2 u, 2 u + 1; tiles past the last: none) of one operand into stages t % 4:
  // instruction i of wave w fills the stage's chunks (8 i + w) 64 + lane (rows past
  // the sequence read its last row: finite, and masked to p = 0).  A row's offset inside its
  // tile fits 32 bits: with nq <= 65535 (attn_args) a row is at most 50.4 MB, 64 rows 3.2 GB.
  const unsigned rowb = (unsigned)(ROW * (int64_t)sizeof(f16));
  const unsigned chunk = (unsigned)(((lane & 15) ^ swz16(4 * wave + (lane >> 4))) << 4);
  const unsigned off0 = (unsigned)(4 * wave + (lane >> 4)) * rowb + chunk;
  auto issue = [&](uint64_t base, f16* ring, int u) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int t = 2 * u + b;
      if (t >= n_tiles) continue;
      const uint64_t tb = base + (uint64_t)(t * kBN) * rowb;
      const int rows = seqlen - 1 - t * kBN;
      const unsigned last = (unsigned)(rows < kBN ? rows : kBN) * rowb + chunk;   // kBN: none clamped
#pragma unroll
      for (int i = 0; i < kFLoads; ++i) {
        const unsigned off = off0 + (unsigned)(32 * i) * rowb;
        const int dst = (t % kFwdStages) * kTileHalves + (8 * i + wave) * 512;
        dma16s(tb, off < last ? off : last, __builtin_amdgcn_readfirstlane(lds_addr(ring + dst)));
      }
    }
  };
  issue(kbase, Ks, 0);
  // this lane's query row as the B operand (rows past the sequence: zeros).  Loaded at a clamped
  // row unconditionally and selected at once, so the compiler's wait for these loads stands here
  // (it then also covers the first K pair, issued above) and not inside the loop.
  f16x8 qf[kHD / 16];
  {
    const f16* qrow = a.qkv + (s0 + (mval ? m : mstart)) * ROW + h * kHD + 8 * hl;
#pragma unroll
    for (int s = 0; s < kHD / 16; ++s) qf[s] = *reinterpret_cast<const f16x8*>(qrow + 16 * s);
    // (the empty asm needs the loaded values: the compiler can neither predicate the loads on
    // mval nor defer their wait into the loop)
#pragma unroll
    for (int s = 0; s < kHD / 16; ++s) asm volatile("" : "+v"(qf[s]));
#pragma unroll
    for (int s = 0; s < kHD / 16; ++s) qf[s] = mval ? qf[s] : zero8();
  }
  wait_vmem<0>();
  issue(vbase, Vs, 0);
  issue(kbase, Ks, 1);
  __syncthreads();
  const unsigned krow = lds_addr(Ks) + row_base(lane), vcol = lds_addr(Vs) + col_base(lane);
  // S^T = K Q^T of tile t: keys kb * 32 + (row of the result), queries on the lanes
  auto scores = [&](f32x16 (&sc)[2], int t) {
    const unsigned ka = fresh(krow + (unsigned)((t % kFwdStages) * kTileHalves * 2));
    sc[0] = sc[1] = zero16();
#pragma unroll
    for (int s = 0; s < kHD / 16; ++s)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        sc[kb] = mfma(lds_read8(ka ^ (unsigned)(32 * s), kb * 32 * kHD * 2), qf[s], sc[kb]);
  };
  f32x16 sc[2], sn[2];
  if (kg < n_tiles) scores(sc, kg);
  wait_vmem<0>();
  __syncthreads();
  // tile t, whose scores are in sc: its softmax and O^T += V^T P^T, beside the scores of tile
  // t + 2 into sn when there is one.  DIAG: the tile may hold masked keys (past this lane's query or
  // the sequence end): key n = n0 + off + 4 (l / 32) is kept iff
  // off <= min(m, seqlen - 1) - n0 - 4 (l / 32).  A lane can see a tile whose keys are all masked
  // before any kept key (this wave skips every other tile): masked probabilities are set to 0
  // rather than computed from the running maximum.
  auto tile = [&](int t, bool more, f32x16 (&sc)[2], f32x16 (&sn)[2], auto diag_c) {
    constexpr bool DIAG = decltype(diag_c)::value;
    const unsigned va = fresh(vcol + (unsigned)((t % kFwdStages) * kTileHalves * 2));
    const int lim = (m < seqlen - 1 ? m : seqlen - 1) - t * kBN - 4 * hl;
    if constexpr (DIAG) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          sc[kb][v] = kb * 32 + 8 * (v >> 2) + (v & 3) <= lim ? sc[kb][v] : -1.0e30f;
    }
    // the row maximum of the raw scores, scaled once (the scaling is monotonic)
    float mx = -1.0e30f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int v = 0; v < 16; ++v) mx = fmaxf(mx, sc[kb][v]);
    mx = half_max(mx);
    // m_i is the reference point of l_i and O, not the exact running maximum: it moves (and O
    // and l are rescaled) only when some lane's maximum exceeds it by more than 2^8, so p =
    // 2^(s * qk_scale - m_i) stays below 256 and the rescale, a read-modify-write of all of O,
    // runs on the first tile and rarely after.  The decision is per wave (uniform branch).
    const float mt = __fmul_rn(mx, a.qk_scale);
    if (__builtin_amdgcn_ballot_w64(mt > m_i + 8.0f) != 0) {
      const float m_new = fmaxf(m_i, mt);
      const float alpha = ex2(__fsub_rn(m_i, m_new));
      l_i = __fmul_rn(l_i, alpha);
      m_i = m_new;
#pragma unroll
      for (int hb = 0; hb < kHD / 32; ++hb)
#pragma unroll
        for (int v = 0; v < 16; ++v) oacc[hb][v] = __fmul_rn(oacc[hb][v], alpha);
    }
    if (!DIAG || more) scores(sn, t + 2);
    float rs[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    f16x8 pf[kBN / 16];   // P^T as the B operand: keys 16 tt .. + 15
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        float p = ex2(__builtin_fmaf(sc[kb][v], a.qk_scale, -m_i));
        if constexpr (DIAG) p = kb * 32 + 8 * (v >> 2) + (v & 3) <= lim ? p : 0.0f;
        rs[v & 3] = __fadd_rn(rs[v & 3], p);
        pf[2 * kb + (v >> 3)][v & 7] = (f16)p;
      }
    l_i = __fadd_rn(l_i, __fadd_rn(__fadd_rn(rs[0], rs[1]), __fadd_rn(rs[2], rs[3])));
    // O^T += V^T P^T over the tile's 64 keys, 16 per step
#pragma unroll
    for (int tt = 0; tt < kBN / 16; ++tt)
#pragma unroll
      for (int hb = 0; hb < kHD / 32; ++hb)
        oacc[hb] = mfma(lds_col8(va, hb, 16 * tt * kHD * 2), pf[tt], oacc[hb]);
    // the next tile's scores spread over the exponentials, their operands read four MFMAs ahead;
    // then O, its operands four MFMAs (eight reads) ahead
    if constexpr (!DIAG) {
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int i = 0; i < 12; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
      }
    } else {
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 200, 0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
  };
  using Diag = std::integral_constant<bool, true>;
  using Full = std::integral_constant<bool, false>;
  // V of pair u and K of pair u + 1 are in LDS; K of pair u + 2 goes where pair u's was (its
  // scores are done), V of pair u + 1 where pair u - 1's was
  auto fetch = [&](int u) {
    issue(vbase, Vs, u + 1);
    issue(kbase, Ks, u + 2);
  };
  // the loads of fetch(u) have landed and are visible, and every wave is done with pair u's V and
  // pair u + 1's K
  auto next = [&]() {
    wait_vmem<0>();
    __syncthreads();
  };
  // pairs whose tiles both lie before the block's first query (no masked key) and have a next
  // tile, two at a time so that the two score buffers need no copies; then the last ones
  int full = mstart / (2 * kBN);
  if (full > (n_tiles - 2) / 2) full = (n_tiles - 2) / 2;
  if (full < 0) full = 0;
  int u = 0;
  for (; u + 2 <= full; u += 2) {
    fetch(u);
    tile(2 * u + kg, true, sc, sn, Full{});
    next();
    fetch(u + 1);
    tile(2 * u + 2 + kg, true, sn, sc, Full{});
    next();
  }
  for (; u < n_pairs; ++u) {
    fetch(u);
    const int t = 2 * u + kg;
    if (t < n_tiles) tile(t, t + 2 < n_tiles, sc, sn, Diag{});
    sc[0] = sn[0];
    sc[1] = sn[1];
    next();
  }
  l_i = __fadd_rn(l_i, __shfl_xor(l_i, 32));
  // merge: the odd-tile wave of each query group hands its state (O lane-major, 16 KB per wave,
  // in the K stages; m and l in the V stages' last KB) to the even-tile wave, which combines
  // O = O0 2^(m0 - m) + O1 2^(m1 - m), l likewise, m = max(m0, m1).  Every stage is free after
  // the loop's last barrier.
  float* ohand = reinterpret_cast<float*>(Ks) + qw * (kHD / 32) * 16 * 64;
  float* mlhand = reinterpret_cast<float*>(Vs) + (kFwdStages * kTileHalves / 2 - 256) + qw * 64;
  static_assert(4 * (kHD / 32) * 16 * 64 * 4 <= kFwdStages * kTileHalves * 2, "O hand-over in Ks");
  if (kg == 1) {
#pragma unroll
    for (int hb = 0; hb < kHD / 32; ++hb)
#pragma unroll
      for (int v = 0; v < 16; ++v) ohand[(hb * 16 + v) * 64 + lane] = oacc[hb][v];
    if (hl == 0) {
      mlhand[c] = m_i;
      mlhand[32 + c] = l_i;
    }
  }
  __syncthreads();
  // result register v of block hb: head column hb * 32 + 8 (v / 4) + 4 (l / 32) + v % 4; one
  // correctly rounded reciprocal per row, then a product per element.  The query group's 32 x 128
  // block of O is staged in the V stages (clear of the hand-over) and written back 16 bytes per
  // lane, four whole 256-byte rows per store instruction.
  constexpr int kOStride = kHD + 8;   // halves per staged row
  static_assert(4 * 32 * kOStride + 512 <= kFwdStages * kTileHalves, "O staging in Vs");
  f16* ostage = Vs + qw * 32 * kOStride;
  if (kg == 0) {
    const float m1 = mlhand[c], l1 = mlhand[32 + c];
    const float mm = fmaxf(m_i, m1);
    const float a0 = ex2(__fsub_rn(m_i, mm)), a1 = ex2(__fsub_rn(m1, mm));
    const float l = __fadd_rn(__fmul_rn(l_i, a0), __fmul_rn(l1, a1));
    const float inv_l = __fdiv_rn(1.0f, l);   // rows past the sequence: not stored
#pragma unroll
    for (int hb = 0; hb < kHD / 32; ++hb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int v = 4 * g + e;
          const float ov = __fadd_rn(__fmul_rn(oacc[hb][v], a0),
                                     __fmul_rn(ohand[(hb * 16 + v) * 64 + lane], a1));
          o[e] = (f16)__fmul_rn(ov, inv_l);
        }
        *reinterpret_cast<f16x4*>(ostage + c * kOStride + hb * 32 + 8 * g + 4 * hl) = o;
      }
    if (mval && hl == 0) lse[(int64_t)h * a.n_tokens + s0 + m] = __fadd_rn(mm, log2f(l));
  }
  __syncthreads();
  // the two waves of a query group store 16 of its 32 rows each
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 16 * kg + 4 * i + (lane >> 4), cc = lane & 15;
    const int row = mstart + 32 * qw + r;
    const f16x8 v = *reinterpret_cast<const f16x8*>(ostage + r * kOStride + 8 * cc);
    if (row < seqlen && s0 + row < a.n_tokens)
      *reinterpret_cast<f16x8*>(out + (s0 + row) * (int64_t)(a.nq * kHD) + h * kHD + 8 * cc) = v;
  }
}

}  // namespace

extern "C" int dk_attn_fwd(const void* qkv, const int32_t* cu_seqlens, int32_t n_seq,
                           const int32_t* block_table, int32_t n_blocks, int64_t n_tokens,
                           int32_t nq, int32_t nkv, int32_t hd, void* out, float* lse,
                           hipStream_t stream) {
  AttnArgs a;
  if (int e = attn_args(a, qkv, cu_seqlens, n_seq, block_table, n_blocks, n_tokens, nq, nkv, hd))
    return e;
  if (n_blocks == 0) return 0;
  if (!out || !lse) return DK_ERR_INVALID;
  if (!dk_aligned(out, 16) || !dk_aligned(lse, 4)) return DK_ERR_ALIGN;
  // the workgroup's index (a token per block at the least: no device holds that many)
  if ((int64_t)n_blocks * nq > INT32_MAX) return DK_ERR_INVALID;
  hipLaunchKernelGGL(attn_fwd_kernel, dim3((unsigned)n_blocks, (unsigned)nq), dim3(kFThreads), 0,
                     stream, a, (f16*)out, lse, n_blocks);
  DK_CHECK_LAUNCH();
  return 0;
}
