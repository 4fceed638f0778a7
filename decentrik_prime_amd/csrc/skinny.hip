// Forward GEMMs of a few rows on gfx950: C[m][n] = sum_k A[m][k] W[n][k] for M <= 32, W stored
// [N][K] as packed NF4 or (F16) already dequantised to fp16; both forms give the same bits.
//
// Bound: reading the packed weight once (0.52 bytes per weight) and converting it (one LDS lookup
// and about five vector instructions per two weights).  The 128-row tiles of w4gemm.hip do the
// work of 128 rows and put 96 to 140 workgroups on the 256 CUs; here a workgroup owns 16 output
// columns (SwiGLU: 16 gate and the same 16 up columns), its KS waves take 256-wide slices of K in
// turn, and every weight is loaded and converted exactly once, straight into the W operand of
// v_mfma_f32_16x16x32_f16 (column l % 16): lane l loads the 64 consecutive weights of its column
// at 256 c + 64 (l / 16), 32 bytes and one first-level block, which are the W operands of eight
// MFMAs whose A operands are the same k of row l % 16.  A slice's loads all go out before the
// previous slice is converted.  The waves' sums meet in LDS, are added in wave order and go
// through the epilogue of the other NF4 GEMMs (the same roundings): no partials in memory, one
// launch.  Measured on MI355X at one row against the 128-row tiles (their reduce launch included):
// gate|up 25 -> 9.1 us, down 23 -> 9.5, a 1536 x 1536 projection 10.5 -> 4.6 (NF4); 25 -> 14,
// 19 -> 13, 8.9 -> 4.2 (fp16).  Up to 16 rows every shape gains (at 16: 25 -> 12.1, 23 -> 14.6,
// 10.9 -> 5.7); with two row tiles only small weights do (skinny_takes): a 1536 x 1536
// projection at 32 rows 11.4 -> 7.5, but fp16 down 20 -> 33.
#include "gemm_common.h"

namespace dk {
namespace {

constexpr int kSliceK = 256;    // K per wave and turn
constexpr int kMaxWaves = 8;

// One slice of one 16-column block: this lane's 64 weights, and for NF4 their scales.
template <bool F16>
struct Slice {
  u32x4 w[F16 ? 8 : 2];
  uint32_t code;
  float s2, o2;
};

template <int EPI, int MT, bool F16>
__global__ __launch_bounds__(64 * kMaxWaves) void skinny_kernel(GemmParams p) {
  constexpr int CB = EPI == EPI_SWIGLU_FWD ? 2 : 1;   // column blocks: gate and up, or one
  __shared__ f32x2 pair_lut[256];   // byte -> (NF4[high nibble], NF4[low nibble])
  __shared__ float c2t[256];
  __shared__ __attribute__((aligned(16))) float red[kMaxWaves][CB * MT][256];
  const int tid = threadIdx.x, lane = tid & 63, ks = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int64_t M = p.M, K = p.K;
  const int64_t n0 = (int64_t)blockIdx.x * 16;
  const int slices = (int)((K + kSliceK - 1) / kSliceK);
  if constexpr (!F16) {
    for (int i = tid; i < 256; i += (int)blockDim.x) {
      pair_lut[i] = f32x2{p.nf4[i >> 4], p.nf4[i & 15]};
      c2t[i] = p.code2[i];
    }
  }
  int64_t wrow[CB];     // this lane's row of W
  const f16* arow[MT];  // this lane's rows of A (rows past M: the last, never stored)
#pragma unroll
  for (int b = 0; b < CB; ++b) wrow[b] = (n0 + lr + (b ? p.inter : 0)) * K;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int64_t m = 16 * t + lr < M ? 16 * t + lr : M - 1;
    arow[t] = p.a + m * p.lda;
  }
  // slice c: K is a multiple of 64, so a lane's 64 weights lie inside K or past it; past it the
  // last ones are read, and use() sets both operands to zero (in that one slice only)
  auto load = [&](int c, Slice<F16> (&sl)[CB], f16x8 (&a)[MT][8]) {
    const int64_t k0 = (int64_t)c * kSliceK + 64 * lg;
    const int64_t k = k0 < K ? k0 : K - 64;
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const int64_t e = wrow[b] + k;
      if constexpr (F16) {
        const u32x4* src = reinterpret_cast<const u32x4*>(p.w16 + e);
#pragma unroll
        for (int j = 0; j < 8; ++j) sl[b].w[j] = src[j];
        continue;
      }
      const u32x4* src = reinterpret_cast<const u32x4*>(p.packed + (e >> 1));
      sl[b].w[0] = src[0];
      sl[b].w[1] = src[1];
      sl[b].code = p.qabs[e >> 6];
      sl[b].s2 = p.scale2[e >> 14];
      sl[b].o2 = p.offset2[e >> 14];
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int j = 0; j < 8; ++j) a[t][j] = *reinterpret_cast<const f16x8*>(arow[t] + k + 8 * j);
  };
  f32x4 acc[CB][MT];
#pragma unroll
  for (int b = 0; b < CB; ++b)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[b][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto use = [&](int c, Slice<F16> (&sl)[CB], f16x8 (&a)[MT][8]) {
    if ((c + 1) * (int64_t)kSliceK > K) {   // the last, partial slice: lanes past K add 0 * 0
      const bool in = (int64_t)c * kSliceK + 64 * lg < K;
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          a[t][j] = in ? a[t][j] : f16x8{};
#pragma unroll
      for (int b = 0; b < CB; ++b) {
        if constexpr (F16) {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            sl[b].w[j] = in ? sl[b].w[j] : u32x4{0, 0, 0, 0};
        } else {
          sl[b].s2 = in ? sl[b].s2 : 0.0f;
          sl[b].o2 = in ? sl[b].o2 : 0.0f;
        }
      }
    }
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const float amax = F16 ? 0.0f : dk_absmax(c2t[sl[b].code], sl[b].s2, sl[b].o2);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        u32x4 o;
        if constexpr (F16) {
          o = sl[b].w[j];
        } else {
          const uint32_t w = sl[b].w[j >> 2][j & 3];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x2 nv = pair_lut[(w >> (8 * q)) & 0xffu];
            o[q] = dk_pack2(dk_h(__fmul_rn(nv[0], amax)), dk_h(__fmul_rn(nv[1], amax)));
          }
        }
        const f16x8 wf = __builtin_bit_cast(f16x8, o);
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t][j], wf, acc[b][t], 0, 0, 0);
      }
    }
  };
  Slice<F16> s0[CB];
  f16x8 a0[MT][8];
  if constexpr (MT == 1 || !F16) {
    // two slices in registers: the next one's loads go out before this one's conversion
    Slice<F16> s1[CB];
    f16x8 a1[MT][8];
    if (wave < slices) load(wave, s0, a0);
    __syncthreads();   // the tables are filled
    for (int c = wave; c < slices; c += 2 * ks) {
      if (c + ks < slices) load(c + ks, s1, a1);
      use(c, s0, a0);
      if (c + 2 * ks < slices) load(c + 2 * ks, s0, a0);
      if (c + ks < slices) use(c + ks, s1, a1);
    }
  } else {
    // two would not fit: the other waves hide the loads
    __syncthreads();
    for (int c = wave; c < slices; c += ks) {
      load(c, s0, a0);
      use(c, s0, a0);
    }
  }
#pragma unroll
  for (int b = 0; b < CB; ++b)
#pragma unroll
    for (int t = 0; t < MT; ++t)
      *reinterpret_cast<f32x4*>(&red[wave][b * MT + t][4 * lane]) = acc[b][t];
  __syncthreads();
  // register v of lane l: row 4 (l / 16) + v, column l % 16; one wave per 16-row tile
  if (wave >= MT) return;
  for (int t = wave; t < MT; t += ks) {
    f32x4 sum[CB];
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      sum[b] = *reinterpret_cast<const f32x4*>(&red[0][b * MT + t][4 * lane]);
      for (int w = 1; w < ks; ++w) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(&red[w][b * MT + t][4 * lane]);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[b][e] += v[e];
      }
    }
    const int64_t n = n0 + lr;
    if constexpr (EPI == EPI_LINEAR) {
      const float bias = p.bias ? (float)p.bias[n] : 0.0f;
      float res[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) res[v] = (float)dk_h(__fadd_rn(sum[0][v], bias));
      for (int q = 0; q < p.n_lora; ++q) {
        const LoraTerm& L = p.lora[q];
        if (n0 < L.n_begin || n0 >= L.n_end) continue;   // ranges are multiples of 32 columns
        const int64_t zr = 16 * t + lr < M ? 16 * t + lr : M - 1;
        f32x4 lo = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int rc = 0; rc < p.rank; rc += 16) {
          const f16x4 zf = *reinterpret_cast<const f16x4*>(L.z + zr * p.rank + rc + 4 * lg);
          const f16x4 rf = *reinterpret_cast<const f16x4*>(L.r + (n - L.n_begin) * p.rank + rc + 4 * lg);
          lo = __builtin_amdgcn_mfma_f32_16x16x16f16(zf, rf, lo, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)
          res[v] = __fadd_rn(res[v], __fmul_rn(L.scale, (float)dk_h(lo[v])));
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t m = 16 * t + 4 * lg + v;
        if (m < M) reinterpret_cast<f16*>(p.out)[m * p.ldo + n] = dk_h(res[v]);
      }
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t m = 16 * t + 4 * lg + v;
        if (m >= M) continue;
        const f16 g = dk_h(sum[0][v]), u = dk_h(sum[1][v]);
        float sig, silu;
        dk_silu_parts((float)g, &sig, &silu);
        reinterpret_cast<f16*>(p.out)[m * p.ldo + n] = dk_h(silu * (float)u);
        if (p.gu) {
          p.gu[m * 2 * p.inter + n] = g;
          p.gu[m * 2 * p.inter + p.inter + n] = u;
        }
      }
    }
  }
}

}  // namespace

template <int EPI, bool F16>
int skinny_launch(const GemmParams& p, hipStream_t stream) {
  const int64_t cols = EPI == EPI_SWIGLU_FWD ? p.inter : p.N;
  const int64_t blocks = cols / 16, slices = (p.K + kSliceK - 1) / kSliceK;
  // waves per workgroup: up to eight over K while the launch has fewer than eight waves per CU
  // (256 CUs) to keep loads in flight, each with at least one slice
  int ks = 1;
  while (ks < kMaxWaves && 2 * ks <= slices && blocks * ks < 2048) ks *= 2;
  if (blocks <= 0 || blocks > 0x7fffffff) return DK_ERR_INVALID;
  const dim3 grid((unsigned)blocks), block(64 * ks);
  if constexpr (EPI == EPI_LINEAR) {
    if (p.M > 16) {
      hipLaunchKernelGGL((skinny_kernel<EPI, 2, F16>), grid, block, 0, stream, p);
      DK_CHECK_LAUNCH();
      return 0;
    }
  }
  hipLaunchKernelGGL((skinny_kernel<EPI, 1, F16>), grid, block, 0, stream, p);
  DK_CHECK_LAUNCH();
  return 0;
}

template int skinny_launch<EPI_LINEAR, false>(const GemmParams&, hipStream_t);
template int skinny_launch<EPI_SWIGLU_FWD, false>(const GemmParams&, hipStream_t);
template int skinny_launch<EPI_LINEAR, true>(const GemmParams&, hipStream_t);
template int skinny_launch<EPI_SWIGLU_FWD, true>(const GemmParams&, hipStream_t);

}  // namespace dk
